"""What the compiler makes of the kernels that stage rows in LDS behind its back and ask for weights past the end of a block-row.

Requests that may lie past the end of what they read go through buffer resources, whose bounds check counts the vector
offset and the immediate one.  The scalar offset is not part of what the compiler's builtin promises to check: no request
may carry one.

A wait that leaves n requests outstanding stands for the rows in LDS only if n were issued behind the last of those rows, on
every path that leads to it."""
import re
import subprocess

import pytest

from tests import isa_waits
import __graft_entry__ as entry


@pytest.fixture(scope="module")
def assemblies(tmp_path_factory):
    recipe = entry._load_build_recipe()
    flags = [f for f in recipe.DEVICE if not f.startswith("-Rpass")]
    out = {}
    for source in ("f32_sparse.hip", "bsr_linear.hip"):
        to = tmp_path_factory.mktemp("staged") / "out.s"
        subprocess.run([recipe.HIPCC, *recipe.COMMON, *flags, "--offload-device-only", "-S", str(recipe.PKG / "csrc" / source), "-o", str(to)],
                       check=True, capture_output=True)
        out[source] = to.read_text()
    return out


@pytest.mark.parametrize("source,at_least", [("f32_sparse.hip", 3), ("bsr_linear.hip", 9)])
def test_no_request_carries_a_scalar_offset(assemblies, source, at_least):
    seen, bad = set(), []
    for name, (code, _) in isa_waits.kernels(assemblies[source]).items():
        for i in code:
            if i.op.startswith("buffer_load"):
                seen.add(name)
                if not re.match(r"^0( |$)", i.operands[3]):
                    bad.append((name, i.text))
    assert len(seen) >= at_least, sorted(seen)
    assert bad == []


def short_waits(code, labels):
    """(waits in assembly that leave requests outstanding, those of them that fewer requests than that may stand behind the
    last row asked into LDS).  `before`: the least number of requests since such a row over all paths to an instruction."""
    before, todo, waits = {0: 64}, [0], {}
    while todo:
        at = todo.pop()
        since = before[at]
        ins = code[at]
        if ins.in_asm and ins.op == "s_waitcnt":
            waits.update({at: n <= since for counter, n in ins.waits if counter == "vmcnt" and n})
        if ins.queue == "vmcnt":
            since = 0 if "_load_lds_" in ins.op else min(64, since + 1)
        following = ([] if ins.ends else [at + 1]) + ([labels[ins.target]] if ins.target else [])
        for to in following:
            if to < len(code) and before.get(to, 65) > since:
                before[to] = since
                todo.append(to)
    return len(waits), [code[at].text for at, enough in waits.items() if not enough]


@pytest.mark.parametrize("source,kernel,found", [("f32_sparse.hip", "bsr16_linear_strip_f32_kernel", 1), ("bsr_linear.hip", "bsr16_linear_halves_kernel", 9)])
def test_waits_for_staged_rows_count_what_is_behind_them(assemblies, source, kernel, found):
    kernels = {n: k for n, k in isa_waits.kernels(assemblies[source]).items() if kernel in n}
    assert len(kernels) == found
    for name, (code, labels) in kernels.items():
        waits, short = short_waits(code, labels)
        assert waits and not short, (name, waits, short)
    # a wait that leaves more than that outstanding is seen
    later = re.sub(r"(ASMSTART\s+s_waitcnt vmcnt\()([1-9]\d*)", lambda m: m[1] + str(int(m[2]) + 40), assemblies[source])
    for name, (code, labels) in isa_waits.kernels(later).items():
        assert kernel not in name or short_waits(code, labels)[1], name


def test_a_load_whose_value_nobody_wants_ends_with_its_wait():
    """attention.hip asks for lines in assembly and drops their values: a register the compiler takes as free would be written
    when the line arrives, unless the same block waits for it."""
    source = (entry.PKG_DIR / "csrc" / "attention.hip").read_text()
    blocks = re.findall(r"asm volatile\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)\s*:\s*\"=&?v\"", source)
    loads = [b for b in blocks if "_load_" in b]
    assert loads and all("s_waitcnt vmcnt(0)" in b.split("_load_")[-1] for b in loads), loads
