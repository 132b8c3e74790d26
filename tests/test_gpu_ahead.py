"""Attention launches that ask for later launches' weights on the way (et_mha_fused_ahead_f16): the attention is the same to
the bit, whichever form runs it and however the spans are cut; what the entry refuses."""
import ctypes as C

import numpy as np
import pytest

from tests import harness as Hn

pytestmark = pytest.mark.gpu

up = Hn.up


class Span(C.Structure):
    _fields_ = [("data", C.c_void_p), ("bytes", C.c_size_t)]


def spans(*of):
    return (Span * len(of))(*of)


# pad 4, rows of the result off 16 bytes: one, two, four and eight waves, two tiles a wave, waves in turn with whole and ragged strips; pad 0: few short sequences
# the same, the others in the 32 x 32 kernel; heads of 32 to 200
SHAPES = [(1, 16, 2, 32, False), (3, 32, 4, 64, True), (2, 128, 12, 64, False), (32, 128, 12, 64, False), (64, 256, 8, 64, False), (16, 512, 8, 64, True),
          (2, 64, 4, 200, False), (16, 128, 16, 64, False), (3, 1296, 12, 64, False), (16, 256, 12, 32, False)]


@pytest.mark.parametrize("B,S,nh,hd,causal", SHAPES)
@pytest.mark.parametrize("pad", [0, 4])
@pytest.mark.parametrize("sizes", [(127,), (128,), (128 * 1000 + 64,), (0, 300, 128 * 77, 128 * 5000)])
def test_ahead_changes_nothing(et, B, S, nh, hd, causal, sizes, pad):
    H, T = nh * hd, B * S
    qkv, weights = up(et, Hn.randn((T, 3 * H), 1)), [up(et, np.full(max(n, 4) // 4, 7, np.int32)) for n in sizes]
    lens = up(et, np.array([S - 3 * (b % 4) for b in range(B)], np.int32))
    got = []
    for ahead in (None, spans(*[(w.ptr, w.nbytes if n else 0) for w, n in zip(weights, sizes)])):
        z = up(et, np.full((T, H + pad), 7.0, np.float16))
        et.check(et.lib().et_mha_fused_ahead_f16(qkv.ptr, qkv.ptr + 2 * H, qkv.ptr + 4 * H, 3 * H, 3 * H, 3 * H, z.ptr, H + pad, None, lens.ptr, B, S, nh,
                                                 hd, hd ** -0.5, et.MHA_CAUSAL if causal else 0, ahead, len(sizes) if ahead else 0, None))
        got.append(z.numpy().view(np.uint16))
    assert np.array_equal(*got)


def test_refusals(et):
    z = et.DeviceBuffer.empty((16, 64), np.float16)

    def status(ahead, n):
        return et.lib().et_mha_fused_ahead_f16(z.ptr, z.ptr, z.ptr, 64, 64, 64, z.ptr, 64, None, None, 1, 16, 1, 64, 0.125, 0, ahead, n, None)

    ok = (z.ptr, 256)
    assert status(spans(ok), 1) == 0
    for ahead, n in ((None, 1), (spans(ok), -1), (spans(ok, ok, ok, ok, ok), 5), (spans((None, 256)), 1), (spans((z.ptr + 2, 256)), 1),
                     (spans((z.ptr, 1 << 31)), 1)):
        assert status(ahead, n) != 0, n
