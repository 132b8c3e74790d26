"""Attention on products of 32 x 32: every form of the rule against attention in binary64, at the edges of its tiles, and the forms that
results off 16-byte alignment keep."""
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

from tests import harness as Hn

ROOT = Path(__file__).resolve().parent.parent
T41, T81, T42, T82, T44 = (4, 1, 2), (8, 1, 2), (4, 2, 2), (8, 2, 2), (4, 4, 1)
# sequences, keys, heads, head size, causal, lengths, the form: whole and cut blocks, heads narrower than their template, tiles without
# queries, sequences of no keys
SHAPES = [
    (70, 16, 12, 64, False, None, T41), (40, 48, 12, 40, True, None, T41), (64, 128, 12, 64, False, [0, 1, 63, 64, 65, 127], T41),
    (8, 784, 12, 64, True, [784, 3, 33, 783], T41), (16, 400, 16, 64, True, None, T81), (20, 176, 12, 64, False, [176, 129, 128, 31], T81),
    (32, 272, 12, 64, False, [272, 129, 128, 31], T81),
    (1, 400, 12, 56, False, None, T44), (3, 528, 12, 64, True, [390, 5], T44), (1, 528, 12, 64, False, [515], T42), (2, 1040, 12, 64, True, None, T42),
    (2, 784, 16, 64, False, [784, 130], T42), (2, 784, 16, 64, False, None, T82),
    # sequences of no keys whose tiles are shared
    (3, 400, 16, 64, False, [400, 77, 0], T42), (3, 784, 10, 88, False, [784, 77, 0], T82), (3, 528, 12, 64, True, [528, 77, 0], T44), (3, 528, 12, 24, False, [528, 77, 0], T42),
    (3, 400, 8, 128, False, [400, 77, 0], T42), (3, 272, 4, 200, False, [272, 77, 0], (4, 2, 1)),
    (20, 512, 12, 32, False, [512, 100, 0], T41), (3, 400, 12, 24, True, None, T44), (4, 272, 12, 32, False, None, T42),
    (8, 272, 10, 80, False, [272, 75, 0], T41), (8, 400, 10, 96, True, None, T81), (1, 400, 10, 80, False, None, T42), (3, 784, 10, 88, False, None, T82),
    (4, 528, 8, 128, False, [528, 513, 7], T41), (12, 272, 8, 120, True, None, T81), (1, 400, 8, 128, False, [399], T44), (2, 1040, 8, 128, True, None, T42),
    (3, 16, 4, 200, True, [16, 1, 0], (4, 1, 1)), (2, 272, 4, 200, False, [272, 65], (4, 2, 1)), (8, 784, 4, 224, False, None, T41),
    (8, 784, 4, 136, True, None, T81), (2, 1552, 4, 136, True, None, (4, 2, 1)),
]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("tiles") / "attention_tiles"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", str(ROOT / "scpaper-2021_amd" / "csrc"), str(ROOT / "tests" / "cpp" / "attention_tiles.cpp"),
                    "-o", str(exe)], check=True)

    def answers(shapes):  # (sequences, keys, heads, head size, causal, lengths)
        text = "\n".join(f"{next(t for t in (32, 64, 96, 128, 224, 256) if hd <= t)} {S} {B * nh} {int(c)} {B if any(lens or ()) else 0}"
                         for B, S, nh, hd, c, *lens in shapes)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        return [tuple(map(int, line.split())) for line in out]

    return answers


def test_the_shapes_run_what_they_claim(ask):
    assert ask([s[:6] for s in SHAPES]) == [s[6] for s in SHAPES]
    assert {(64, f) for f in (T41, T81, T42, T82, T44)} <= {(s[3], s[6]) for s in SHAPES}


def test_what_the_one_launch_with_projection_takes_keeps_its_bits(ask):
    """Few short sequences run the kernel that the launch joined with the projection is made of; heads beyond 224 too."""
    assert ask([(1, 128, 12, 64, False), (8, 128, 12, 64, True), (1, 384, 12, 64, False), (5, 256, 8, 128, False), (12, 96, 4, 256, False)]) == [(0, 0, 0)] * 5


def test_wide_causal_heads_take_the_form_measured_fastest(ask):
    """One strip of eight waves is as long as its longest wave: two waves a tile where the chip is not full, and the other kernel for 65 to 96 keys."""
    T421 = (4, 2, 1)
    assert ask([(1, 1536, 4, 200, True), (2, 2048, 4, 200, True), (1, 2048, 6, 136, True)]) == [T421] * 3
    assert ask([(8, 2048, 4, 200, True), (4, 3072, 4, 200, True)]) == [T81] * 2
    assert ask([(1, 80, 4, 200, True), (24, 80, 5, 160, True), (8, 96, 6, 136, True)]) == [(0, 0, 0)] * 3
    assert ask([(24, 80, 6, 136, True), (16, 96, 4, 200, True), (1, 80, 4, 200, False)]) == [(4, 1, 1)] * 3


def test_sequences_of_their_own_lengths_keep_four_waves_where_eight_are_few(ask):
    few = [(4, 640, 16, 64, False), (3, 784, 12, 64, False), (4, 512, 16, 64, False), (8, 400, 12, 64, False), (4, 1024, 10, 80, False), (8, 512, 10, 80, False)]
    assert [w for w, *_ in ask(few)] == [8] * 6
    assert [w for w, *_ in ask([(*s, [1]) for s in few])] == [4] * 6
    alone = [(1, 2048, 12, 64, False), (1, 3584, 10, 80, False)]  # one sequence has nothing to even out
    assert ask([(*s, [1]) for s in alone]) == ask(alone) and [w for w, *_ in ask(alone)] == [8] * 2
    many = [(16, 2048, 12, 64, False, [1]), (8, 1024, 16, 64, False, [1]), (3, 1536, 8, 128, False, [1]), (3, 784, 10, 88, False, [1])]
    assert [w for w, *_ in ask(many)] == [8] * 4


def test_few_long_sequences_keep_the_form_measured_fastest(ask):
    """One workgroup of eight waves a unit, heads of 64: ahead of two of four; from 2560 keys on whole strips keep the waves in turn."""
    assert ask([(4, 1024, 16, 64, False), (4, 1280, 12, 64, False), (2, 2048, 16, 64, False), (1, 8192, 12, 64, False)]) == [T81] * 4
    assert ask([(1, 4096, 12, 64, False), (1, 3584, 16, 64, False), (1, 3072, 16, 64, False), (1, 4096, 16, 64, False, [1])]) == [(0, 0, 0)] * 4
    assert ask([(1, 4080, 12, 64, False), (2, 6144, 8, 64, False), (2, 2048, 16, 64, False, [1]), (16, 2048, 16, 64, False)]) == [T81, T41, T41, T81]


def test_causal_strips_that_meet_on_a_unit_keep_the_form_measured_fastest(ask):
    assert ask([(4, 1024, 16, 64, True), (5, 1024, 12, 64, True), (2, 2048, 16, 64, True), (7, 448, 10, 80, True)]) == [T41, T41, T42, T81]
    assert ask([(1, 4096, 16, 64, True), (1, 1024, 16, 64, True)]) == [T82, T44]


def test_few_wide_heads_of_padded_short_sequences_keep_the_other_kernel(ask):
    assert ask([(1, 80, 4, 200, False, [1]), (5, 80, 6, 136, False, [1])]) == [(0, 0, 0)] * 2
    assert ask([(8, 80, 4, 200, False, [1]), (5, 80, 6, 136, False)]) == [(4, 1, 1)] * 2


def test_four_workgroups_of_shared_tiles_a_unit_are_one_too_many(ask):
    assert ask([(12, 208, 12, 32, False), (12, 224, 12, 32, False, [1])]) == [T42] * 2
    assert ask([(1, 400, 12, 32, False)]) == [T44]


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,nh,hd,causal,lens,form", SHAPES)
@pytest.mark.parametrize("pad", [0, 4])
def test_against_binary64(et, B, S, nh, hd, causal, lens, form, pad):
    """pad 4: rows of the result 8-byte aligned only, which the 32 x 32 kernel does not take.  Bound: the probabilities enter the product
    rounded to binary16 (2^-11 each, against a row sum of those same values) and so does the result: 2^-10 of max |V| < 5.5, with as much again for the
    binary32 sums."""
    H, T = nh * hd, B * S
    qkv = Hn.randn((T, 3 * H), 5)
    n = [S] * B if lens is None else [lens[b % len(lens)] for b in range(B)]
    if B > 1:
        qkv[S:2 * S] = np.nan  # a sequence that holds no number: its neighbours do not depend on it
    d, d_l = Hn.up(et, qkv), Hn.up(et, np.array(n, np.int32)) if lens is not None else None
    d_z = Hn.up(et, np.full((T, H + pad), 7.0, np.float16))
    et.mha_fused(d.ptr, d.offset(2 * H), d.offset(4 * H), 3 * H, 3 * H, 3 * H, d_z.ptr, H + pad, None, None if d_l is None else d_l.ptr, B, S, nh, hd,
                 hd ** -0.5, et.MHA_CAUSAL if causal else 0, None)
    got = d_z.numpy()
    assert np.all(got[:, H:] == 7.0)
    for b in sorted({0, 2, 3, 4, 5, B - 1} & set(range(B)) - {1}):
        x = torch.from_numpy(qkv[b * S:(b + 1) * S].astype(np.float64)).view(S, 3, nh, hd).permute(1, 2, 0, 3).contiguous()
        s = torch.matmul(x[0], x[1].transpose(1, 2).contiguous()) * hd ** -0.5
        s[:, :, n[b]:] = -np.inf
        if causal:
            s.masked_fill_(torch.ones(S, S, dtype=torch.bool).triu(1), -np.inf)
        want = torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), x[2]).transpose(0, 1).reshape(S, H).numpy()
        assert np.abs(got[b * S:(b + 1) * S, :H] - want).max() <= 1.1e-2
        assert np.linalg.norm(got[b * S:(b + 1) * S, :H] - want) <= 5e-4 * np.linalg.norm(want)


# sequences, keys, heads, head size, causal, the form; the first column of a block of 64 keys, and the second, are where a length ends
PADDED = [(64, 128, 12, 64, True, T41), (30, 272, 12, 64, False, T81), (1, 528, 12, 64, False, T42), (3, 784, 10, 88, False, T82), (3, 528, 12, 64, True, T44),
          (20, 512, 12, 32, True, T41), (8, 272, 10, 80, True, T41), (4, 528, 8, 128, False, T41), (8, 784, 4, 224, False, T41)]


def test_the_padded_shapes_run_what_they_claim(ask):
    assert ask([(*s[:5], [1]) for s in PADDED]) == [s[5] for s in PADDED]


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,nh,hd,causal,form", PADDED)
@pytest.mark.parametrize("length", [1, 32, 65, 96])
def test_rows_past_a_length_need_hold_no_numbers(et, B, S, nh, hd, causal, form, length):
    """Rows of K and V from the next multiple of 32 past a sequence's length on are no numbers, and no result depends on them.  Bound as above."""
    H, T = nh * hd, B * S
    qkv = Hn.randn((T, 3 * H), 7).reshape(B, S, 3, H)
    qkv[:, (length + 31) // 32 * 32:, 1:] = np.nan
    d, d_l, d_z = Hn.up(et, qkv), Hn.up(et, np.full(B, length, np.int32)), Hn.up(et, np.full((T, H), 7.0, np.float16))
    et.mha_fused(d.ptr, d.offset(2 * H), d.offset(4 * H), 3 * H, 3 * H, 3 * H, d_z.ptr, H, None, d_l.ptr, B, S, nh, hd, hd ** -0.5, et.MHA_CAUSAL if causal else 0, None)
    got = d_z.numpy().reshape(B, S, H)
    for b in sorted({0, B - 1}):
        x = torch.from_numpy(qkv[b].astype(np.float64)).view(S, 3, nh, hd).permute(1, 2, 0, 3).contiguous()
        s = torch.matmul(x[0], x[1][:, :length].transpose(1, 2).contiguous()) * hd ** -0.5
        if causal:
            s.masked_fill_(torch.ones(S, length, dtype=torch.bool).triu(1), -np.inf)
        want = torch.matmul(torch.softmax(s, -1), x[2][:, :length]).transpose(0, 1).reshape(S, H).numpy()
        assert np.abs(got[b] - want).max() <= 1.1e-2
        assert np.linalg.norm(got[b] - want) <= 5e-4 * np.linalg.norm(want)
