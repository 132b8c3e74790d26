"""The token-local launches of an encoder layer (et_encoder_layer_f32: output projection, LayerNorm, FFN, LayerNorm and
the next QKV projection of a strip of token rows in one workgroup, or in several that share the strip) against the
binary32 mathematics of the same steps."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import layers as L
from tests import harness as Hn
from tests.harness import up

pytestmark = pytest.mark.gpu


class Weights(C.Structure):
    """et_layer_weights of include/et_abi.h"""
    _fields_ = [(n, C.c_void_p * 4) for n in ("row_ptr", "col_idx", "tiles", "bias")] + [(n, C.c_void_p * 2) for n in ("gamma", "beta")]


def tile_order(x):
    """[T x H] -> tile order: 16 tokens x 16 features together, token r, features 4g .. 4g + 3 at 4 (16 g + r)."""
    T, H = x.shape
    return np.ascontiguousarray(x.reshape(T // 16, 16, H // 16, 4, 4).transpose(0, 2, 3, 1, 4))


def row_order(t, T, H):
    return np.ascontiguousarray(t.reshape(T // 16, H // 16, 4, 16, 4).transpose(0, 3, 1, 2, 4)).reshape(T, H)


# widths at the edges: one block-row per wave and fewer (16, 48, 240, 256), two to four with waves that hold one less
# (272, 384, 800), the widest; hidden widths of one block-row, of one chunk, of several; 16 to 80 rows so that a 32-row
# strip ends in half a strip; shares that divide the block-rows and that do not; empty and nearly full weights
CASES = [(16, 16, 16, 1, 1, 0.0), (48, 48, 32, 2, 1, 0.5), (240, 256, 80, 1, 3, 0.7), (256, 1024, 16, 1, 7, 0.95),
         (272, 208, 48, 2, 1, 0.8), (384, 1536, 64, 1, 4, 0.6), (768, 3072, 48, 1, 1, 0.8), (768, 3072, 80, 2, 1, 0.8),
         (768, 3072, 32, 1, 5, 0.9), (800, 208, 48, 1, 2, 0.3), (800, 208, 48, 2, 1, 0.6), (1024, 4096, 48, 2, 1, 0.9),
         (1024, 4096, 32, 1, 12, 0.95), (1024, 4096, 16, 1, 1, 0.1)]


@pytest.mark.parametrize("H,FF,T,mt,parts,sparsity", CASES)
@pytest.mark.parametrize("project,act", [(True, 2), (False, 1)])
def test_token_local_layer(et, H, FF, T, mt, parts, sparsity, project, act):
    lib = et.lib()
    Q = 3 * H if project else 0
    mats = [Hn.BsrWeight(o, i, sparsity, seed=31 + k, std=0.05, bias_std=0.1)
            for k, (o, i) in enumerate(((H, H), (FF, H), (H, FF), (3 * H, H)))]
    norms = [Hn.randn((H,), 60 + k, 0.1) for k in range(4)]
    norms[0], norms[2] = norms[0] + np.float16(1), norms[2] + np.float16(1)
    Z, x16 = Hn.randn((T, H), 70), Hn.randn((T, H), 71)
    x32 = Hn.randn((T, H), 72, dtype=np.float32)
    w, keep = Weights(), []
    for k, m in enumerate(mats):
        for name, arr in (("row_ptr", m.row_ptr), ("col_idx", m.col_idx if len(m.col_idx) else np.zeros(1, np.int32)),
                          ("tiles", m.tiles if len(m.tiles) else np.zeros((1, 256), np.float16)), ("bias", m.bias)):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
    for k in range(2):
        for name, arr in (("gamma", norms[2 * k]), ("beta", norms[2 * k + 1])):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
    assert lib.et_encoder_layer_supported(T, H, FF, Q) == 1
    pack = C.c_void_p()
    et.check(lib.et_encoder_layer_pack_create(C.byref(w), T, H, FF, Q, mt, parts, C.byref(pack)))
    dZ, d16 = up(et, Z), up(et, x16)
    f = Hn.f32

    def half(t):  # what a matrix-core operand is rounded to
        return t.to(torch.float16).float()

    for wide in (True, False):
        d32 = up(et, tile_order(x32))
        o32 = et.DeviceBuffer.empty((T, H), np.float32)
        o16 = et.DeviceBuffer.empty((T, H), np.float16)
        qkv = et.DeviceBuffer.empty((T, 3 * H), np.float16)
        partial = et.DeviceBuffer.empty((parts, T, H), np.float32)
        for _ in range(2):  # the second run on what the first left in the workspace
            et.check(lib.et_encoder_layer_f32(pack, dZ.ptr, d32.ptr if wide else None, None if wide else d16.ptr, o32.ptr, o16.ptr,
                                              qkv.ptr if Q else None, partial.ptr, act, 1e-5, 1e-5, None))
        x = torch.from_numpy(x32) if wide else f(x16)

        def norm(v, k):
            return torch.nn.functional.layer_norm(v, (H,), f(norms[2 * k]), f(norms[2 * k + 1]), 1e-5)

        def lin(v, m):
            return v @ f(m.dense).T + f(m.bias)

        y = norm(lin(f(Z), mats[0]) + x, 0)
        h = lin(half(y), mats[1])
        h = torch.relu(h) if act == 1 else torch.nn.functional.gelu(h, approximate="tanh")
        want = norm(lin(half(h), mats[2]) + y, 1)
        got = torch.from_numpy(row_order(o32.numpy(), T, H).copy())
        # the hidden operand's rounding (2^-11 of its values) may fall the other way where the sums differ in their last
        # bits: relative error of the layer's result well below one binary16 unit
        assert torch.norm(got - want) / torch.norm(want) <= 2e-4
        assert Hn.max_abs(o16.numpy(), got.numpy()) <= 4e-3
        if Q:
            want_q = lin(half(got), mats[3])
            assert torch.norm(f(qkv.numpy()) - want_q) / torch.norm(want_q) <= 5e-4
    et.check(lib.et_encoder_layer_pack_destroy(pack))


@pytest.mark.parametrize("H,nh,FF,S,B,sparsity,mixed", [(256, 4, 512, 32, 3, 0.7, 1), (768, 12, 512, 112, 7, 0.8, 0),
                                                        (384, 6, 1536, 16, 1, 0.9, 1), (128, 2, 256, 16, 270, 0.6, 1)])
def test_stacks_on_token_local_launches(et, H, nh, FF, S, B, sparsity, mixed):
    """Stacks the engine runs this way by itself (48 to 4320 rows: shared strips, one workgroup a strip, 32-row strips):
    graph and eager the same bits, in place, and near the oracle."""
    layers = [Hn.LayerWeights(H, nh, FF, sparsity, seed=800 + i) for i in range(3)]
    lens = np.random.default_rng(S).integers(S // 2, S + 1, B).astype(np.int32)
    x = Hn.randn((B * S, H), 811)
    outs = []
    for use_graph in (True, False):
        m = Hn.build_model(et, layers, S, B, lens=lens, mixed=mixed, use_graph=use_graph)
        assert m.launches_per_layer() == 2  # attention, and the token-local part in one launch, whether or not strips are shared
        d = et.DeviceBuffer.from_numpy(x)
        o = et.DeviceBuffer.empty(x.shape, np.float16)
        m.forward(o, d)
        m.sync()
        outs.append(o.numpy())
        m.forward(d, d)
        m.sync()
        outs.append(d.numpy())
    for o in outs[1:]:
        assert np.array_equal(outs[0], o)
    want = Hn.oracle_stack(x, layers, B, lens, store=torch.float16, resid=torch.float32 if mixed else "same")
    a, b = outs[0].astype(np.float32), want.astype(np.float32)
    for i in range(B):
        a[i * S + lens[i]:(i + 1) * S] = 0
        b[i * S + lens[i]:(i + 1) * S] = 0
    # binary32 residual: one binary16 unit at |x| <= 4 and noise, as for the other forms of it; a binary16 one is rounded
    # in every layer, and the oracle rounds the two projections ahead of it besides
    assert Hn.max_abs(a, b) <= (4e-3 if mixed else 2e-2)


def test_token_local_refusals(et):
    lib, w, pack = et.lib(), Weights(), C.c_void_p()
    assert lib.et_encoder_layer_supported(32, 1040, 256, 0) == 0 and lib.et_encoder_layer_supported(24, 256, 256, 0) == 0
    assert lib.et_encoder_layer_supported(32, 256, 4112, 0) == 0 and lib.et_encoder_layer_supported(32, 256, 256, 3088) == 0
    assert lib.et_encoder_layer_pack_create(C.byref(w), 32, 256, 256, 0, 1, 1, C.byref(pack)) == et.ET_ERR_INVALID_ARG
    assert lib.et_encoder_layer_pack_create(C.byref(w), 32, 256, 256, 0, 2, 2, C.byref(pack)) == et.ET_ERR_INVALID_ARG
    assert lib.et_encoder_layer_pack_create(None, 32, 256, 256, 0, 1, 1, C.byref(pack)) == et.ET_ERR_INVALID_ARG
    assert lib.et_encoder_layer_f32(None, None, None, None, None, None, None, None, 0, 1e-5, 1e-5, None) == et.ET_ERR_INVALID_ARG


def layer_pack(et, T, H, FF, parts, tiles_of_first_row=None):
    """(status, pack, what has to stay alive) of a layer without projection; the first block-row of Wo may be given as that
    many tiles on column 0."""
    w, keep, pack = Weights(), [], C.c_void_p()
    for k, (o, i) in enumerate(((H, H), (FF, H), (H, FF))):
        m = Hn.BsrWeight(o, i, 0.5, seed=91 + k, std=0.01, bias_std=0.1)
        row_ptr, col_idx, tiles = m.row_ptr, m.col_idx, m.tiles
        if k == 0 and tiles_of_first_row is not None:
            first = int(row_ptr[1])
            row_ptr = np.concatenate([row_ptr[:1], row_ptr[1:] - first + tiles_of_first_row]).astype(np.int32)
            col_idx = np.concatenate([np.zeros(tiles_of_first_row, np.int32), col_idx[first:]])
            tiles = np.concatenate([Hn.randn((tiles_of_first_row, 256), 97, 0.01), tiles[first:]])
        for name, arr in (("row_ptr", row_ptr), ("col_idx", col_idx), ("tiles", tiles), ("bias", m.bias)):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
        keep.append((row_ptr, col_idx, tiles, m.bias))
    for k in range(2):
        for name, arr in (("gamma", np.ones(H, np.float16)), ("beta", np.zeros(H, np.float16))):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
    return et.lib().et_encoder_layer_pack_create(C.byref(w), T, H, FF, 0, 1, parts, C.byref(pack)), pack, keep, w


def test_token_local_longest_block_row(et):
    """A descriptor counts up to 255 slots of two tiles: 510 tiles in a block-row (columns may occur more than once) are
    multiplied, 511 have no pack."""
    T, H, FF = 32, 48, 32
    st, pack, _, _ = layer_pack(et, T, H, FF, 1, 511)
    assert st == et.ET_ERR_UNSUPPORTED and not pack.value
    st, pack, keep, _ = layer_pack(et, T, H, FF, 1, 510)
    et.check(st)
    mats = [k for k in keep if isinstance(k, tuple)]

    def dense(m, n_in):  # tiles of one position add up
        d = torch.zeros(16 * (len(m[0]) - 1), n_in)
        for r in range(len(m[0]) - 1):
            for t in range(m[0][r], m[0][r + 1]):
                d[16 * r:16 * r + 16, 16 * m[1][t]:16 * m[1][t] + 16] += torch.from_numpy(m[2][t].astype(np.float32)).view(16, 16)
        return d

    Z, x = Hn.randn((T, H), 98), Hn.randn((T, H), 99)
    out = et.DeviceBuffer.empty((T, H), np.float16)
    dZ, dx = up(et, Z), up(et, x)
    et.check(et.lib().et_encoder_layer_f32(pack, dZ.ptr, None, dx.ptr, None, out.ptr, None, None, 0, 1e-5, 1e-5, None))
    f, norm = Hn.f32, lambda v: torch.nn.functional.layer_norm(v, (H,), eps=1e-5)
    y = norm(f(Z) @ dense(mats[0], H).T + f(mats[0][3]) + f(x))
    h = (y.half().float() @ dense(mats[1], H).T + f(mats[1][3])).half().float()
    want = norm(h @ dense(mats[2], FF).T + f(mats[2][3]) + y)
    assert Hn.max_abs(out.numpy(), want.numpy()) <= 4e-3
    et.check(et.lib().et_encoder_layer_pack_destroy(pack))


def test_token_local_refuses_addresses_and_overlap(et):
    """Before any launch: buffers off the addresses the kernel's loads and stores need, and a result over the residual."""
    lib, T, H, FF, parts = et.lib(), 32, 48, 32, 2
    st, pack, keep, w = layer_pack(et, T, H, FF, parts)
    et.check(st)
    half, wide = T * H * 2, T * H * 4
    buf = et.DeviceBuffer.empty((4 * half + 8 * wide,), np.uint8)
    Z, x16, out16 = buf.ptr, buf.ptr + half + 64, buf.ptr + 2 * half + 128
    x32 = buf.ptr + 4 * half
    o32, partial = x32 + wide, x32 + 2 * wide

    def call(Z=Z, x32=x32, x16=None, o32=o32, out16=out16, partial=partial):
        return lib.et_encoder_layer_f32(pack, Z, x32, x16, o32, out16, None, partial, 0, 1e-5, 1e-5, None)

    for bad in (dict(Z=Z + 8), dict(x32=x32 + 4), dict(o32=o32 + 8), dict(partial=partial + 4), dict(out16=out16 + 4),
                dict(x32=None, x16=x16 + 4)):
        assert call(**bad) == et.ET_ERR_UNSUPPORTED, bad
    for bad in (dict(o32=x32), dict(o32=x32 + 16), dict(o32=x32 + wide - 16, partial=partial + wide), dict(o32=x32 - wide + 16)):
        assert call(**bad) == et.ET_ERR_INVALID_ARG, bad
    w.tiles[1] = w.tiles[1] + 8
    other = C.c_void_p()
    assert lib.et_encoder_layer_pack_create(C.byref(w), T, H, FF, 0, 1, parts, C.byref(other)) == et.ET_ERR_UNSUPPORTED
    assert lib.et_encoder_layer_project_f16(pack, x16, Z, None) == et.ET_ERR_UNSUPPORTED  # no projection in the pack
    assert lib.et_encoder_layer_project_f16(pack, None, Z, None) == et.ET_ERR_INVALID_ARG
    et.check(lib.et_encoder_layer_pack_destroy(pack))


@pytest.mark.parametrize("H,FF,T,mt,parts,sparsity", [
    (16, 32, 16, 1, 2, 0.0), (48, 80, 48, 1, 3, 0.5), (272, 208, 144, 1, 4, 0.8), (768, 3072, 80, 1, 7, 0.9), (1024, 4096, 32, 1, 12, 0.6),
    (48, 32, 48, 2, 1, 0.5), (384, 1536, 64, 1, 1, 0.6), (768, 3072, 80, 2, 1, 0.8), (1024, 4096, 48, 2, 1, 0.9)])
def test_projection_alone_repeats_the_launches(et, H, FF, T, mt, parts, sparsity):
    """QKV made from the rounded result on its own: the bits the launches of the layer left, and the Linear of that result
    (as test_token_local_layer bounds it).  Packs of one part have such a launch only when asked for it."""
    lib, w, keep, pack = et.lib(), Weights(), [], C.c_void_p()
    mats = [Hn.BsrWeight(o, i, sparsity, seed=31 + k, std=0.05, bias_std=0.1) for k, (o, i) in enumerate(((H, H), (FF, H), (H, FF), (3 * H, H)))]
    for k, m in enumerate(mats):
        for name, arr in (("row_ptr", m.row_ptr), ("col_idx", m.col_idx), ("tiles", m.tiles), ("bias", m.bias)):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
    for k in range(2):
        for name, arr in (("gamma", np.ones(H, np.float16)), ("beta", np.zeros(H, np.float16))):
            keep.append(up(et, arr))
            getattr(w, name)[k] = keep[-1].ptr
    et.check(lib.et_encoder_layer_pack_create_projecting(C.byref(w), T, H, FF, 3 * H, mt, parts, C.byref(pack)))
    Z, x = up(et, Hn.randn((T, H), 70)), up(et, Hn.randn((T, H), 71))
    out, partial = et.DeviceBuffer.empty((T, H), np.float16), et.DeviceBuffer.empty((parts, T, H), np.float32)
    qkv = [et.DeviceBuffer.from_numpy(np.full((T, 3 * H), np.nan, np.float16)) for _ in range(2)]
    et.check(lib.et_encoder_layer_f32(pack, Z.ptr, None, x.ptr, None, out.ptr, qkv[0].ptr, partial.ptr, 2, 1e-5, 1e-5, None))
    et.check(lib.et_encoder_layer_project_f16(pack, out.ptr, qkv[1].ptr, None))
    assert np.array_equal(qkv[0].numpy(), qkv[1].numpy())
    want = Hn.f32(out.numpy()) @ Hn.f32(mats[3].dense).T + Hn.f32(mats[3].bias)
    assert torch.norm(Hn.f32(qkv[1].numpy()) - want) / torch.norm(want) <= 5e-4
    et.check(lib.et_encoder_layer_pack_destroy(pack))
    et.check(lib.et_encoder_layer_pack_create(C.byref(w), T, H, FF, 3 * H, 1, 1, C.byref(pack)))
    assert lib.et_encoder_layer_project_f16(pack, out.ptr, qkv[1].ptr, None) == et.ET_ERR_UNSUPPORTED
    et.check(lib.et_encoder_layer_pack_destroy(pack))


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("use_graph", [True, False])
def test_token_local_stack_at_any_address(et, mixed, use_graph):
    """A model takes its input and result where the separate launches took them: the input four bytes, the result two off
    the alignment of the token-local launches, the same bits as at aligned addresses, on every replay."""
    H, nh, FF, S, B = 256, 4, 512, 64, 5
    layers = [Hn.LayerWeights(H, nh, FF, 0.7, seed=830 + i) for i in range(5)]
    m = Hn.build_model(et, layers, S, B, mixed=mixed, use_graph=use_graph)
    assert m.launches_per_layer() == 2
    x = Hn.randn((B * S, H), 831)
    want = et.DeviceBuffer.empty(x.shape, np.float16)
    d = et.DeviceBuffer.from_numpy(x)
    m.forward(want, d)
    m.sync()
    shifted_in = et.DeviceBuffer.from_numpy(np.concatenate([np.zeros(2, np.float16), x.reshape(-1)]))
    shifted_out = et.DeviceBuffer.from_numpy(np.zeros(x.size + 1, np.float16))
    for _ in range(3):
        m.forward(shifted_out.ptr + 2, shifted_in.ptr + 4)
        m.sync()
        assert np.array_equal(shifted_out.numpy(np.float16, (x.size + 1,))[1:].reshape(x.shape), want.numpy())
        et.check(et.lib().et_fill_f16(shifted_out.ptr, x.size + 1, 0x7E00, None))
        et.sync()
