"""Both parts of a shared strip in one launch (et_encoder_layer_joined_f32) against the two launches of the same pack: the same
bits, whether the workgroups of a strip wait for each other (their meeting bounded by `spin`) or leave their share of the
projection to the last of them at once (spin = 0)."""
import ctypes as C

import numpy as np
import pytest

from tests import harness as Hn
from tests.harness import up
from tests.test_gpu_encoder_layer import Weights, tile_order

pytestmark = pytest.mark.gpu


def make_pack(et, H, FF, T, parts, sparsity, project):
    w, keep = Weights(), []

    def put(name, k, arr):
        keep.append(up(et, arr))
        getattr(w, name)[k] = keep[-1].ptr

    for k, (o, i) in enumerate(((H, H), (FF, H), (H, FF), (3 * H, H))):
        m = Hn.BsrWeight(o, i, sparsity, seed=31 + k, std=0.05, bias_std=0.1)
        for name, arr in (("row_ptr", m.row_ptr), ("col_idx", m.col_idx), ("tiles", m.tiles), ("bias", m.bias)):
            put(name, k, arr)
    for k in range(2):
        put("gamma", k, Hn.randn((H,), 60 + k, 0.1) + np.float16(1))
        put("beta", k, Hn.randn((H,), 63 + k, 0.1))
    pack = C.c_void_p()
    et.check(et.lib().et_encoder_layer_pack_create(C.byref(w), T, H, FF, 3 * H if project else 0, 1, parts, C.byref(pack)))
    return pack, keep


# two to four block-rows a wave and fewer waves with any; parts that divide nothing, one to nine strips (more than one on an
# XCD), 2 to 12 parts
@pytest.mark.parametrize("H,FF,T,parts", [(256, 1024, 16, 7), (384, 1536, 144, 4), (400, 208, 48, 2), (768, 3072, 128, 8), (768, 3072, 1040, 3),
                                          (1024, 4096, 32, 12), (1024, 2048, 80, 2)])
@pytest.mark.parametrize("project", [True, False])
def test_joined_equals_two_launches(et, H, FF, T, parts, project):
    lib = et.lib()
    pack, keep = make_pack(et, H, FF, T, parts, 0.8, project)
    joins = C.c_int()
    et.check(lib.et_encoder_layer_joins(pack, C.byref(joins)))
    assert joins.value == 1
    Z, x16, x32 = up(et, Hn.randn((T, H), 70)), up(et, Hn.randn((T, H), 71)), up(et, tile_order(Hn.randn((T, H), 72, dtype=np.float32)))
    partial, words = et.DeviceBuffer.empty((parts, T, H), np.float32), up(et, np.zeros(T // 16, np.int32))

    def outputs(run, wide):
        o32, o16 = et.DeviceBuffer.empty((T, H), np.float32), et.DeviceBuffer.empty((T, H), np.float16)
        qkv = up(et, np.zeros((T, 3 * H), np.float16))
        et.check(run(pack, Z.ptr, x32.ptr if wide else None, None if wide else x16.ptr, o32.ptr, o16.ptr, qkv.ptr if project else None, partial.ptr))
        return [b.numpy().view(np.uint8) for b in (o32, o16, qkv)]

    for wide in (True, False):
        want = outputs(lambda *a: lib.et_encoder_layer_f32(*a, 2, 1e-5, 1e-5, None), wide)
        for spin in (4000, 0, 1, 4000):
            got = outputs(lambda *a: lib.et_encoder_layer_joined_f32(*a, words.ptr, spin, 2, 1e-5, 1e-5, None), wide)
            assert all(np.array_equal(a, b) for a, b in zip(got, want)), (wide, spin)
            assert not words.numpy().any()
    et.check(lib.et_encoder_layer_pack_destroy(pack))


def test_joined_refusals(et):
    lib = et.lib()
    H, FF, T = 256, 512, 32
    pack, keep = make_pack(et, H, FF, T, 2, 0.8, False)
    one, keep1 = make_pack(et, H, FF, T, 1, 0.8, False)
    b = [et.DeviceBuffer.empty((4, T, H), np.float32) for _ in range(4)]
    words = up(et, np.zeros(T // 16, np.int32))

    def status(p, join, spin, partial=b[3].ptr):
        return lib.et_encoder_layer_joined_f32(p, b[0].ptr, None, b[1].ptr, b[2].ptr, None, None, partial, join, spin, 2, 1e-5, 1e-5, None)

    assert status(pack, words.ptr, 10) == 0
    joins = C.c_int(1)
    et.check(lib.et_encoder_layer_joins(one, C.byref(joins)))
    assert joins.value == 0
    for p, join, spin, partial in ((one, words.ptr, 10, b[3].ptr), (pack, None, 10, b[3].ptr), (pack, words.ptr + 2, 10, b[3].ptr), (pack, words.ptr, -1, b[3].ptr),
                                   (pack, words.ptr, 10, None)):
        assert status(p, join, spin, partial) != 0
    et.sync()
    for p in (pack, one):
        et.check(lib.et_encoder_layer_pack_destroy(p))
