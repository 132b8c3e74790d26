"""The rules that choose a kernel's form (csrc/*_forms.h), asked on the host: what the tests of the forms claim to run, and
where the lines between them lie."""
import subprocess
from pathlib import Path

import pytest

from tests import test_gpu_ahead as ahead
from tests import test_gpu_attention_variants as attention
from tests import test_gpu_kernels as kernels
from tests import test_gpu_linear_formats as linear

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("forms") / "launch_forms"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", str(ROOT / "scpaper-2021_amd" / "csrc"),
                    str(ROOT / "tests" / "cpp" / "launch_forms.cpp"), "-o", str(exe)], check=True)

    def answers(questions):
        res = subprocess.run([str(exe)], input="\n".join(questions) + "\n", capture_output=True, text=True, check=True)
        out = res.stdout.splitlines()
        assert len(out) == len(questions)
        return out

    return answers


def gemm(T, inp, out, batch=1, trans_b=1, dma=1):
    return f"gemm {T} {out} {inp} {batch} {trans_b} {dma}"


def mha(B, S, nh, hd, causal=False, lens=None, compact=False, plain=True, pad=4):
    """pad: halfs between the rows of the result; of 4, they lie off 16 bytes, which the 32 x 32 kernel leaves to the others."""
    HD = next(t for t in (32, 64, 96, 128) if hd <= t)
    return f"mha {HD} {int(compact)} {S} {B * nh} {int(causal)} {int(plain)} {B if lens is not None else 0} {int(pad % 8 == 0)}"


def test_the_dense_tests_run_every_tile(ask):
    got = ask([gemm(*shape) for shape in linear.DMA_FORMS])
    tiles = [(1, 1, 4), (2, 1, 4), (1, 2, 4), (2, 2, 4), (1, 3, 4), (2, 3, 3), (2, 2, 2), (2, 1, 2)]
    forms = {f"tile {a} {b} {n} {ragged}" for a, b, n in tiles for ragged in (0, 1)} | {"tile 4 4 4 0", "tile 4 4 2 1"}
    assert forms - set(got) == {"tile 4 4 2 1"}  # (256 x 256 with ragged edges: test_linear_dense, 8176 x 80 -> 8208)
    assert set(got) - forms == set()
    assert ask([gemm(8176, 80, 8208)]) == ["tile 4 4 2 1"]


def test_rows_off_a_line_run_what_they_claim(ask):
    assert ask([f"lines {T} {out} {inp}" for T, inp, out, _ in linear.LINE_FORMS]) == [tile for *_, tile in linear.LINE_FORMS]
    # two to a compute unit stay where K is short, and where no round is saved and the last is half empty
    assert ask(["lines 5152 1312 496", "lines 1840 3424 912", "lines 1840 3424 1040", "lines 2208 1408 224"]) == ["2 2 2", "2 2 2", "2 2 4", "2 2 4"]


def test_large_dense_problems_keep_tiles_of_256(ask):
    """Edges that are multiples of 64 but not of 256 leave the form of whole tiles as edges of 16 do."""
    large = [(16384, 8192, 8192), (16368, 8192, 8192), (16320, 8192, 8192), (16384, 8192, 8128), (16320, 256, 4096), (8128, 4096, 8256)]
    assert ask([gemm(*shape) for shape in large]) == ["tile 4 4 4 0"] + ["tile 4 4 2 1"] * 5
    assert not any(a.startswith("tile 4 4") for a in ask([gemm(16320, 64, 4096), gemm(8128, 4096, 4032)]))  # too shallow; too few


def test_small_dense_results(ask):
    """Three tiles of 16 x 16 a compute unit, four where the pieces of a wave fill its rounds of loads."""
    small = [(224, 3072, 768), (336, 3072, 768), (256, 784, 768), (512, 256, 512), (352, 768, 704), (176, 1040, 1072), (256, 3088, 768)]
    assert ask([gemm(*shape) for shape in small]) == ["small"] * len(small)
    larger = [(352, 3072, 768), (272, 3088, 768), (784, 2816, 256), (272, 784, 768), (528, 256, 512), (1040, 768, 256), (400, 240, 16)]
    assert "small" not in ask([gemm(*shape) for shape in larger])
    assert ask([gemm(448, 3088, 1008, dma=0), gemm(512, 3088, 1024, dma=0)]) == ["small", "none"]
    assert ask([gemm(256, 2048, 640, batch=2), gemm(272, 2048, 640, batch=2)]) == ["small", "tile 1 1 4 1"]


def test_large_dense_problems_share_a_compute_unit(ask):
    """Several rounds of 128 x 192 tiles on operands out of the caches lose to two workgroups of 128 x 128 a unit; one round of them, and the
    projections of a stack of 2048 rows, keep them."""
    several = [(6000, 3216, 2448), (7104, 2688, 2160), (4736, 2368, 3072), (4992, 2384, 2608)]
    assert all(a.startswith("tile 2 2 2") for a in ask([gemm(*shape) for shape in several]))
    assert ask([gemm(2048, 768, 3072), gemm(2048, 768, 2304)]) == ["tile 2 3 3 0"] * 2


def test_the_ragged_attention_tests_run_what_they_claim(ask):
    shapes = [s for s in attention.RAGGED_STRIPS if s[3] <= 128]
    got = dict(zip([s[:5] for s in shapes], ask([mha(*s) for s in shapes])))
    assert [s[1] for s in shapes if got[s[:5]] == "turns 1"] == [1296, 1296, 912, 1904, 1296]
    assert set(got.values()) == {"turns 1", "waves 8 1", "waves 8 2", "waves 4 1", "waves 2 1", "waves 1 1"}
    assert got[(80, 16, 12, 64, False)] == got[(38, 96, 12, 32, True)] == "waves 2 1" and got[(150, 16, 12, 32, True)] == "waves 1 1"
    assert got[(16, 80, 16, 64, False)] == got[(16, 112, 16, 128, False)] == got[(2, 1024, 16, 128, False)] == got[(16, 256, 8, 128, True)] == "waves 8 1"
    assert got[(64, 32, 8, 32, False)] == "waves 2 1"
    assert got[(40, 512, 16, 88, False)] == "waves 8 2"
    aligned = ask([mha(*s, pad=0) for s in shapes])  # the same with rows of the result at 16 bytes: the 32 x 32 kernel, but for few short sequences
    assert [a.startswith("tiles") for a in aligned] == [S > 384 or B * nh * ((S + 31) // 32) > 400 for B, S, nh, *_ in shapes]


def test_the_attention_tests_run_every_form_of_both_kernels(ask):
    def form(HD, *args, **kw):
        return [(HD, a) for a in ask([mha(*args, **kw)])]

    run = set()
    for B, S, nh, hd, causal, lens in attention.RAGGED_STRIPS:
        if hd <= 128:
            run |= set(form(next(t for t in (32, 64, 96, 128) if hd <= t), B, S, nh, hd, causal, lens))
    for B, S, nh, hd, causal in kernels.LARGE_GRIDS:
        run |= set(form(hd, B, S, nh, hd, causal, [1]))
    for B, S, nh, hd, causal in kernels.MASKED:
        run |= set(form(next(t for t in (32, 64, 96, 128) if hd <= t), B, S, nh, hd, causal, plain=False))
    assert run >= {(HD, f"waves {w}") for HD, ws in ((32, ("4 1", "2 1", "1 1")), (64, ("8 2", "8 1", "4 1", "2 1")), (96, ("8 2", "8 1", "4 1")),
                                                     (128, ("8 1", "4 1", "2 1"))) for w in ws} | {(64, "turns 0"), (64, "turns 1")}
    behind = {a for B, S, nh, hd, causal in ahead.SHAPES if hd <= 64 for a in ask([mha(B, S, nh, hd, causal, [1])])}
    assert behind == {"turns 0", "turns 1", "waves 8 2", "waves 8 1", "waves 4 1"} | (behind & {"waves 2 1", "waves 1 1"})
    assert ask([mha(32, 256, 16, 64, plain=False, pad=0), mha(32, 256, 16, 64, pad=0)]) == ["waves 8 2", "tiles 8 1 2"]


def test_attention_takes_eight_waves_where_they_save_a_unit_time(ask):
    eight = [(16, 128, 16, 64), (16, 256, 8, 64), (17, 640, 8, 128), (8, 896, 16, 128), (2, 1024, 16, 128), (64, 224, 16, 64),
             (54, 96, 16, 64), (66, 96, 8, 64), (59, 80, 16, 40)]  # (the last row: two or three waves without queries)
    four = [(22, 704, 12, 40), (10, 832, 12, 40), (11, 1088, 8, 128), (8, 656, 12, 64), (64, 144, 12, 64), (2, 1024, 10, 80), (44, 128, 16, 128), (54, 128, 16, 64),
            (1, 2048, 8, 128)]  # (the last: 128 workgroups of 8 waves)
    causal8 = [(16, 256, 8, 128), (4, 1152, 12, 64), (6, 896, 12, 64), (64, 128, 12, 64), (10, 1392, 8, 128)]
    causal4 = [(25, 448, 10, 80), (14, 1216, 16, 128), (16, 576, 16, 128), (3, 1152, 12, 64), (8, 896, 12, 64), (40, 256, 10, 96)]
    assert ask([mha(*s) for s in eight]) == ["waves 8 1"] * len(eight)
    assert ask([mha(*s) for s in four]) == ["waves 4 1"] * len(four)
    assert ask([mha(4, 512, 16, 64), mha(4, 512, 16, 64, lens=[1]), mha(8, 256, 16, 64, lens=[1])]) == ["waves 8 1", "waves 4 1", "waves 8 1"]
    uneven8, uneven4 = [(3, 928, 16, 128), (11, 496, 8, 128), (13, 1008, 6, 128)], [(38, 448, 8, 128), (39, 320, 8, 128), (52, 288, 8, 128), (271, 96, 6, 128)]
    assert ask([mha(*s, lens=[1]) for s in uneven8 + uneven4]) == ["waves 8 1"] * 3 + ["waves 4 1"] * 4
    assert ask([mha(*s, True) for s in causal8]) == ["waves 8 1"] * len(causal8)
    assert ask([mha(*s, True) for s in causal4]) == ["waves 4 1"] * len(causal4)
    assert ask([mha(48, 256, 12, 64, True), mha(48, 512, 12, 64, True, plain=False), mha(48, 256, 12, 64)]) == ["waves 8 1", "waves 8 2", "waves 8 2"]


def test_heads_of_128_take_one_tile_a_wave(ask):
    shapes = [(B, S, nh, 128, causal) for B in (1, 16, 32, 47) for nh in (8, 16) for S in range(256, 2049, 256) for causal in (False, True) if B * nh * (S // 256) >= 512]
    for lens in (None, [1]):
        assert set(ask([mha(*s, lens=lens) for s in shapes])) == {"waves 8 1"}


def test_many_short_sequences_take_the_fewest_rounds(ask):
    compact = ask([mha(*s[:4], compact=True) for s in attention.COMPACT_SHAPES])
    assert compact == ["waves 4 1"] * 3 + ["waves 2 1", "waves 2 1", "waves 1 1", "waves 2 1", "waves 4 1"]
    heads64 = {768: 4, 769: 2, 1024: 2, 1025: 4, 1536: 4, 1537: 2, 2049: 4}
    assert ask([mha(n, 16, 1, 64) for n in heads64]) == [f"waves {w} 1" for w in heads64.values()]
    heads32 = {768: 4, 769: 2, 1536: 2, 1537: 1, 2048: 1, 3072: 1}
    assert ask([mha(n, 16, 1, 32) for n in heads32]) == [f"waves {w} 1" for w in heads32.values()]
    assert ask([mha(300, 96, 1, 64), mha(400, 96, 1, 32), mha(560, 96, 1, 32), mha(300, 80, 1, 64, compact=True)]) == \
        ["waves 4 1", "waves 2 1", "waves 4 1", "waves 4 1"]


def test_heads_of_256_take_wide_blocks_alone_on_a_unit(ask):
    assert ask(["wide 640 6", "wide 2048 8", "wide 208 56", "wide 256 64"]) == ["128"] * 4
    assert ask(["wide 192 6", "wide 2064 8", "wide 256 65", "wide 1040 24"]) == ["64"] * 4
    used = [f"wide {S} {B * nh}" for B, S, nh, hd, *_ in attention.RAGGED_STRIPS if hd > 224]
    assert set(ask(used)) == {"64", "128"}


def test_no_causal_or_masked_problem_takes_turns_with_ragged_strips(ask):
    """The ragged form in turns has no causal limits, and neither form adds a mask."""
    shapes = [(B, S, nh, 64) for B in (1, 2, 5, 16) for nh in (12, 16, 31) for S in range(16, 2064, 16)]
    assert "turns 1" in ask([mha(*s) for s in shapes])
    assert "turns 1" not in ask([mha(*s, True) for s in shapes])
    assert not any(a.startswith("turns") for a in ask([mha(*s, plain=False) for s in shapes]))
