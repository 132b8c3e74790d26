"""The native library loads without a GPU and exports every symbol the headers include/*.h declare."""
import ctypes
import re
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def declared_symbols():
    text = "\n".join(h.read_text() for h in sorted((ROOT / "include").glob("*.h")))  # et_abi.h, et_tuning.h
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)  # comments cite names that are not declarations
    return sorted(set(re.findall(r"\b(et_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_surface():
    names = declared_symbols()
    for must in ("et_linear_bsr16_f16", "et_mha_fused_f16", "et_skip_layernorm_f16", "et_model_forward",
                 "et_linear_dense_f16", "et_linear_rowpruned_f16", "et_linear_colpruned_f16",
                 "et_linear_vec1x16_f16", "et_vec1x16_to_dense_f16", "et_linear_csr_f16", "et_mha_compactv_f16", "et_mha_vo_f16",
                 "et_fmt_dense_to_bsr16", "et_graph_launch"):
        assert must in names
    assert len(names) >= 70


def test_library_exports_every_declared_symbol(et):
    lib = et.lib()
    missing = [n for n in declared_symbols() if not hasattr(lib, n)]
    assert missing == []


def test_binding_has_argtypes_for_every_declared_symbol(et):
    untyped = [n for n in declared_symbols()
               if n not in et._SIGNATURES and n not in ("et_status_string", "et_last_error", "et_set_last_error")]
    assert untyped == []


def test_status_strings_and_error_channel(et):
    lib = et.lib()
    assert lib.et_status_string(0) == b"ok"
    assert b"unsupported" in lib.et_status_string(et.ET_ERR_UNSUPPORTED)
    lib.et_set_last_error.argtypes = [ctypes.c_char_p]
    lib.et_set_last_error(b"probe message")
    assert lib.et_last_error() == b"probe message"
    # a host-side entry point fails with a status and a message, never aborts
    n = ctypes.c_int()
    st = lib.et_fmt_tile_pattern(30, 64, 0.5, 1, None, None, ctypes.byref(n))
    assert st == et.ET_ERR_INVALID_ARG and b"multiples of 16" in lib.et_last_error()


def test_no_product_file_imports_the_oracle():
    """The oracle is test infrastructure: nothing under the package or include/ may use it."""
    offenders = []
    for path in list((ROOT / "scpaper-2021_amd").rglob("*")) + list((ROOT / "include").rglob("*")):
        if path.is_file() and path.suffix in (".py", ".h", ".hpp", ".hip", ".cpp") and "build" not in path.parts:
            if re.search(r"^\s*(from|import)\s+oracle\b|oracle/", path.read_text(), flags=re.M):
                offenders.append(str(path))
    assert offenders == []


def test_hot_path_kernels_keep_their_registers():
    """The build records registers, spills and scratch of every kernel next to the library.  A kernel that
    spills vector registers to scratch memory pays for it on every launch (the 12-wave forms of the
    tile-sparse Linear sit at the 168-register limit), so none may.  Scalar registers parked in the lanes of a vector register ("SGPRs Spill") cost a
    v_readlane each and no memory access; the compiler reserves 36 bytes of scratch for such kernels without
    ever addressing it, which is why the criterion is the vector spill count and not the scratch size."""
    import re
    from pathlib import Path
    rec = Path(__file__).resolve().parents[1] / "scpaper-2021_amd" / "lib" / "kernel_resources.txt"
    if not rec.exists():
        pytest.skip("no resource record: the library was built by an older build script")
    seen = 0
    for line in rec.read_text().splitlines():
        m = re.search(r"VGPRs Spill: (\d+)", line)
        sc = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if not m or not sc:
            continue
        seen += 1
        name = line.split()[1]
        vspill, scratch = int(m.group(1)), int(sc.group(1))
        if vspill:
            raise AssertionError(f"{name} spills {vspill} vector registers ({scratch} bytes of scratch per lane)")
        # scratch without vector spills: only the unused reservation that comes with parked scalar registers
        assert scratch <= 36 and (scratch == 0 or int(re.search(r"SGPRs Spill: (\d+)", line).group(1)) > 0), line
        if "bsr16_linear_kernel" in name or "bsr16_packed_kernel" in name or "bsr16_chain_kernel" in name or \
                "mha_fused_kernelILi64ELb0ELi4ELi1E" in name:
            assert vspill == 0 and scratch == 0, line
    assert seen > 100


def test_four_wave_attention_holds_three_waves_a_simd():
    """The four-wave forms that fetch a block ahead are made for three workgroups a compute unit, also where some of their workgroups ask
    for later launches' weights."""
    import re
    from pathlib import Path
    rec = Path(__file__).resolve().parents[1] / "scpaper-2021_amd" / "lib" / "kernel_resources.txt"
    if not rec.exists():
        pytest.skip("no resource record: the library was built by an older build script")
    held = {}
    for line in rec.read_text().splitlines():
        m = re.search(r"mha_fused_(kernelILi(?:32|64)ELb0ELi4ELi1|ahead_kernelILi(?:32|64)ELi4ELi1)E.*Occupancy \[waves/SIMD\]: (\d+)", line)
        if m:
            held[m.group(1)] = int(m.group(2))
    assert len(held) == 4 and min(held.values()) >= 3, held


def test_wide_layernorm_holds_three_waves_a_simd():
    """Binary16 rows of 2049 to 4096 columns without a residual: sixteen chunks a lane, gamma and beta beside them."""
    import re
    from pathlib import Path
    rec = Path(__file__).resolve().parents[1] / "scpaper-2021_amd" / "lib" / "kernel_resources.txt"
    if not rec.exists():
        pytest.skip("no resource record: the library was built by an older build script")
    held = [int(m.group(1)) for m in (re.search(r"layernorm_rows_\w*kernelIDF16_Li16ELb0E.*Occupancy \[waves/SIMD\]: (\d+)", line) for line in rec.read_text().splitlines()) if m]
    assert held == [3], held
