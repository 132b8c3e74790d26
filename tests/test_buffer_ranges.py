"""Requests that may lie past the end of what they read go through buffer resources, whose bounds check counts the vector
offset and the immediate one.  The scalar offset is not part of what the compiler's builtin promises to check: no request
may carry one."""
import re
import subprocess

import pytest

from tests import isa_waits
import __graft_entry__ as entry


@pytest.mark.parametrize("source,at_least", [("f32_sparse.hip", 3), ("bsr_linear.hip", 9)])
def test_no_request_carries_a_scalar_offset(tmp_path, source, at_least):
    recipe = entry._load_build_recipe()
    out = tmp_path / "out.s"
    flags = [f for f in recipe.DEVICE if not f.startswith("-Rpass")]
    subprocess.run([recipe.HIPCC, *recipe.COMMON, *flags, "--offload-device-only", "-S", str(recipe.PKG / "csrc" / source), "-o", str(out)],
                   check=True, capture_output=True)
    seen, bad = set(), []
    for name, (code, _) in isa_waits.kernels(out.read_text()).items():
        for i in code:
            if i.op.startswith("buffer_load"):
                seen.add(name)
                if not re.match(r"^0( |$)", i.operands[3]):
                    bad.append((name, i.text))
    assert len(seen) >= at_least, sorted(seen)
    assert bad == []
