"""GPU parity of the kernel-level C ABI against the CPU oracle (same seeded
inputs).  fp16 path: max-abs <= 2e-2 is the bar the engine is built to; the
per-kernel tests below hold tighter bounds where the arithmetic allows."""
import math

import numpy as np
import pytest
import torch

from oracle import formats as F
from oracle import layers as L
from tests import harness as Hn

pytestmark = pytest.mark.gpu

TOL_F16 = 2e-2


up = Hn.up


# ---------------------------------------------------------------- runtime ----

def test_device_is_gfx950(et):
    info = et.device_info()
    print(info)
    assert "gfx950" in info["name"]
    assert info["num_cu"] >= 1


def test_fill_convert_roundtrip(et):
    n = 100003
    src = Hn.randn((n,), 3, 3.0, np.float32)
    d_src = up(et, src)
    d_h = et.DeviceBuffer.empty((n,), np.float16)
    et.check(et.lib().et_f32_to_f16(d_h.ptr, d_src.ptr, n, None))
    got = d_h.numpy()
    assert np.array_equal(got.view(np.uint16), src.astype(np.float16).view(np.uint16))  # RN-even, bit exact
    d_f = et.DeviceBuffer.empty((n,), np.float32)
    et.check(et.lib().et_f16_to_f32(d_f.ptr, d_h.ptr, n, None))
    assert np.array_equal(d_f.numpy(), got.astype(np.float32))
    et.check(et.lib().et_fill_f16(d_h.ptr, n, int(np.float16(0.2).view(np.uint16)), None))
    assert np.all(d_h.numpy() == np.float16(0.2))
    et.check(et.lib().et_memset(d_h.ptr, 0, n * 2, None))
    assert np.all(d_h.numpy().view(np.uint16) == 0)
    fresh = et.DeviceBuffer.empty((4096,), np.float16)  # et_malloc zero-fills (CUDA_ptr(size))
    assert np.all(fresh.numpy().view(np.uint16) == 0)


# ---------------------------------------------------------------- norms ------

def test_device_memory_comes_from_slabs_and_private_scopes(et):
    """Buffers allocated one after the other lie next to one another (4 KiB granules of a 64 MiB slab), a
    request above a quarter of a slab gets an allocation of its own, a private scope cuts from slabs of its
    own starting at the distance asked for, memory is zero-filled, and everything can be freed in any order."""
    import ctypes as C
    lib = et.lib()
    def alloc(n):
        p = C.c_void_p()
        et.check(lib.et_malloc(C.byref(p), n))
        return p.value
    a, b, c = alloc(100), alloc(5000), alloc(1 << 20)
    assert b - a == 4096 and c - b == 8192
    big = alloc(17 << 20)
    d = alloc(64)
    assert d - c == 1 << 20 and not (a <= big < a + (64 << 20))
    et.check(lib.et_pool_private_begin(3 * 4096))
    p1, p2 = alloc(64), alloc(64)
    assert lib.et_pool_private_begin(0) == et.ET_ERR_INVALID_ARG  # scopes do not nest
    et.check(lib.et_pool_private_end())
    assert lib.et_pool_private_end() == et.ET_ERR_INVALID_ARG
    assert lib.et_pool_private_begin(100) == et.ET_ERR_INVALID_ARG   # not a multiple of 4096
    e = alloc(64)
    assert p2 - p1 == 4096 and p1 % (2 << 20) == 3 * 4096 and abs(p1 - a) >= (32 << 20) and e - d == 4096
    host = np.empty(5000, np.uint8)
    et.check(lib.et_memcpy_d2h(host.ctypes.data, b, 5000))
    assert not host.any()
    for p in (c, p1, a, big, e, b, p2, d):
        et.check(lib.et_free(p))


@pytest.mark.parametrize("rows,H", [(1024, 768), (2048, 1024), (128, 800), (7, 64), (33, 2048), (5, 4100)])
def test_skip_layernorm(et, rows, H):
    src, skip = Hn.randn((rows, H), 1), Hn.randn((rows, H), 2)
    gamma = (1 + Hn.randn((H,), 3, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((H,), 4, 0.1)
    d_out = et.DeviceBuffer.empty((rows, H), np.float16)
    et.skip_layernorm(d_out, up(et, src), up(et, skip), up(et, gamma), up(et, beta), rows, H, 1e-5)
    want = L.skip_layernorm(Hn.f32(src), Hn.f32(skip), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    # one fp16 rounding of an O(4) value: half an ulp = 2e-3
    assert Hn.max_abs(d_out.numpy(), want.numpy()) <= 4e-3


@pytest.mark.parametrize("rows,H", [(1024, 768), (2048, 1024), (128, 800), (7, 64), (5, 4100)])
def test_skip_layernorm_mixed(et, rows, H):
    """binary32 in (a projection's output and the residual), binary32 and binary16 out."""
    src, skip = Hn.randn((rows, H), 1, 0.5, np.float32), Hn.randn((rows, H), 2, 1.0, np.float32)
    gamma = (1 + Hn.randn((H,), 3, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((H,), 4, 0.1)
    d32, d16 = et.DeviceBuffer.empty((rows, H), np.float32), et.DeviceBuffer.empty((rows, H), np.float16)
    args = (up(et, src).ptr, up(et, skip).ptr, up(et, gamma).ptr, up(et, beta).ptr, rows, H, 1e-5, None)
    et.check(et.lib().et_skip_layernorm_mixed(d32.ptr, d16.ptr, *args))
    want = L.skip_layernorm(Hn.f32(src), Hn.f32(skip), Hn.f32(gamma), Hn.f32(beta), 1e-5, None).numpy()
    assert want.dtype == np.float32
    got32, got16 = d32.numpy(), d16.numpy()
    assert Hn.max_abs(got32, want) <= 2e-5          # fp32 statistics on both sides
    assert np.array_equal(got16, got32.astype(np.float16))  # the operand copy is the rounded residual
    # either output alone
    e32, e16 = et.DeviceBuffer.empty((rows, H), np.float32), et.DeviceBuffer.empty((rows, H), np.float16)
    et.check(et.lib().et_skip_layernorm_mixed(e32.ptr, None, *args))
    et.check(et.lib().et_skip_layernorm_mixed(None, e16.ptr, *args))
    assert np.array_equal(e32.numpy(), got32) and np.array_equal(e16.numpy(), got16)


@pytest.mark.parametrize("rows,H", [(1024, 768), (16, 1024), (3, 800)])
def test_layernorm(et, rows, H):
    src = Hn.randn((rows, H), 5, 2.0)
    gamma = (1 + Hn.randn((H,), 6, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((H,), 7, 0.1)
    d_out = et.DeviceBuffer.empty((rows, H), np.float16)
    et.layernorm(d_out, up(et, src), up(et, gamma), up(et, beta), rows, H, 1e-5)
    want = L.layernorm(Hn.f32(src), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    assert Hn.max_abs(d_out.numpy(), want.numpy()) <= 4e-3


# rows of up to 512 columns, one or two chunks of four a lane, and the first width that takes three
@pytest.mark.parametrize("rows,H", [(1, 4), (9, 252), (6, 256), (5, 260), (4, 512), (7, 516)])
@pytest.mark.parametrize("skip", [False, True])
def test_layernorm_of_short_rows(et, rows, H, skip):
    """Bound: one binary16 rounding of a value below 8, 2^-9, and the binary32 statistics."""
    src, more = Hn.randn((rows, H), 5, 2.0), Hn.randn((rows, H), 8)
    gamma, beta = (1 + Hn.randn((H,), 6, 0.1, np.float32)).astype(np.float16), Hn.randn((H,), 7, 0.1)
    d_out = up(et, np.full((rows + 1, H), 7.0, np.float16))
    norm = (up(et, gamma), up(et, beta), rows, H, 1e-5)
    if skip:
        et.skip_layernorm(d_out, up(et, src), up(et, more), *norm)
        want = L.skip_layernorm(Hn.f32(src), Hn.f32(more), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    else:
        et.layernorm(d_out, up(et, src), *norm)
        want = L.layernorm(Hn.f32(src), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    got = d_out.numpy()
    assert Hn.max_abs(got[:rows], want.numpy()) <= 4e-3 and (got[rows] == 7.0).all()


# eight chunks a lane and sixteen, their first and last widths, and the first of 32
@pytest.mark.parametrize("rows,H", [(5, 2048), (6, 2052), (1, 3072), (4, 4096), (7, 4100)])
@pytest.mark.parametrize("skip", [False, True])
def test_layernorm_of_wide_rows(et, rows, H, skip):
    test_layernorm_of_short_rows(et, rows, H, skip)


def test_layernorm_rejects_bad_shape(et):
    d = et.DeviceBuffer.empty((16, 16), np.float16)
    st = et.lib().et_layernorm_f16(d.ptr, d.ptr, d.ptr, d.ptr, 4, 6, 1e-5, None)
    assert st == et.ET_ERR_UNSUPPORTED
    st = et.lib().et_skip_layernorm_f16(d.ptr, d.ptr, None, d.ptr, d.ptr, 4, 8, 1e-5, None)
    assert st == et.ET_ERR_INVALID_ARG
    assert b"skip" in et.lib().et_last_error()


# ---------------------------------------------------------------- elementwise

@pytest.mark.parametrize("n", [1024 * 3072, 1000003, 5])
def test_gelu_relu(et, n):
    x = Hn.randn((n,), 8, 2.0)
    d_x = up(et, x)
    d_y = et.DeviceBuffer.empty((n,), np.float16)
    et.check(et.lib().et_gelu_f16(d_y.ptr, d_x.ptr, n, None))
    want = L.gelu_tanh(Hn.f32(x)).half().numpy()
    assert Hn.max_abs(d_y.numpy(), want) <= 2e-3
    et.check(et.lib().et_relu_f16(d_x.ptr, d_x.ptr, n, None))  # in place
    assert np.array_equal(d_x.numpy(), np.maximum(x, np.float16(0)))


@pytest.mark.parametrize("rows,cols", [(128, 768), (33, 50)])
def test_bias_add(et, rows, cols):
    x, b = Hn.randn((rows, cols), 9), Hn.randn((cols,), 10)
    d_x = up(et, x)
    et.check(et.lib().et_bias_add_f16(d_x.ptr, up(et, b).ptr, rows, cols, None))
    want = (x.astype(np.float32) + b.astype(np.float32)).astype(np.float16)
    assert np.array_equal(d_x.numpy().view(np.uint16), want.view(np.uint16))


# ---------------------------------------------------------------- BSR linear -

BSR_CASES = [
    # T, in, out, sparsity, act
    (2048, 768, 768, 0.8, 0),
    (2048, 768, 768, 0.9, 0),
    (2048, 768, 3072, 0.8, 2),
    (2048, 3072, 768, 0.8, 0),
    (1024, 768, 2304, 0.8, 0),
    (128, 800, 208, 0.5, 1),     # the example model's FFN shape (example/main.cu:29)
    (16, 16, 16, 0.0, 0),
    (48, 64, 32, 0.3, 2),
    (2048, 4096, 1024, 0.9, 0),  # BERT-large FFN
    (64, 6144, 64, 0.5, 0),      # input too wide for an LDS-staged strip
    (8192, 768, 768, 0.8, 2),    # enough token rows for 64-row strips
    # launch-geometry paths: 6-wave workgroups (5 and 18 block-rows each), 64-row strips at 4096
    # rows, a ragged last strip with an uneven group split, one block-row per workgroup
    (256, 768, 2304, 0.8, 0),
    (4096, 768, 3072, 0.8, 2),
    (1040, 768, 768, 0.8, 1),
    (16, 768, 3072, 0.8, 0),
    (80, 3072, 768, 0.8, 2),
    # the 90 % rows of the tile-sparse Linear configuration at 2048 token rows
    (2048, 768, 3072, 0.9, 0),
    (2048, 3072, 768, 0.9, 0),
    # unstaged strips (input too wide for LDS) with more block-rows per workgroup than one wave
    # can own before the cap: 320 block-rows, 4 waves
    (16384, 5120, 5120, 0.98, 0),
]


@pytest.mark.parametrize("T,inp,out,sp,act", BSR_CASES)
def test_linear_bsr16(et, T, inp, out, sp, act):
    w = Hn.BsrWeight(out, inp, sp, seed=11, bias_std=0.1).upload(et)
    x = Hn.randn((T, inp), 12)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    w.forward(et, up(et, x), d_y, T, act)
    want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), {0: None, 1: "relu", 2: "gelu"}[act],
                    torch.float16)
    err = Hn.max_abs(d_y.numpy(), want.numpy())
    print(f"bsr T={T} in={inp} out={out} sp={sp}: ntile={len(w.col_idx)} max-abs={err:.2e}")
    # |y| stays below ~4 here: one fp16 rounding (<= 2e-3) plus accumulation-order noise
    assert err <= 4e-3


@pytest.mark.parametrize("strip_rows,inp,out", [(16, 208, 800), (16, 3072, 768), (32, 1024, 528), (64, 768, 2304)])
def test_linear_bsr16_fewer_strips_than_dies(et, strip_rows, inp, out):
    """1 to 9 strips of the height these shapes take, the last one ragged: below 8 strips the workgroups are dealt to the
    dies in runs, from 8 on a strip keeps to one die.  Every value is written, and is that of the oracle."""
    w = Hn.BsrWeight(out, inp, 0.7, seed=21, bias_std=0.1).upload(et)
    for strips in range(1, 10):
        T = strip_rows * strips - (16 if strip_rows > 16 and strips % 2 == 0 else 0)
        x = Hn.randn((T, inp), 22 + strips)
        d_y = up(et, np.full((T, out), np.nan, np.float16))
        w.forward(et, up(et, x), d_y, T, 0)
        want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), None, torch.float16)
        assert Hn.max_abs(d_y.numpy(), want.numpy()) <= 4e-3, (strips, T)


def _random_bsr_cases(n, seed):
    rng = np.random.default_rng(seed)
    cases = []
    for _ in range(n):
        T = 16 * int(rng.integers(1, 25))
        inp = 16 * int(rng.integers(1, 65)) if rng.random() < 0.8 else 16 * int(rng.integers(192, 340))
        out = 16 * int(rng.integers(1, 65)) if rng.random() < 0.8 else 16 * int(rng.integers(100, 200))
        sp = float(rng.choice([0.0, 0.3, 0.5, 0.8, 0.9, 0.97, 1.0]))
        cases.append((T, inp, out, sp, int(rng.integers(0, 3)), int(rng.integers(1, 1 << 30))))
    return cases


@pytest.mark.parametrize("T,inp,out,sp,act,seed", _random_bsr_cases(32, 20211114))
def test_linear_bsr16_random_shapes(et, T, inp, out, sp, act, seed):
    """Seeded random shapes (every launch plan the shape picks: strips of 16, 32 or 64 rows, staged or not, 6, 8
    or 12 waves), binary16 and binary32 result against the oracle."""
    w = Hn.BsrWeight(out, inp, sp, seed=seed, bias_std=0.1).upload(et)
    x = Hn.randn((T, inp), seed ^ 0x5a5a)
    d_x = up(et, x)
    d_y, d_y32 = et.DeviceBuffer.empty((T, out), np.float16), et.DeviceBuffer.empty((T, out), np.float32)
    w.forward(et, d_x, d_y, T, act)
    et.check(et.lib().et_linear_bsr16_f16_f32out(w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, w.d_bias.ptr, d_x.ptr,
                                                d_y32.ptr, T, inp, out, act, None))
    et.sync()
    name = {0: None, 1: "relu", 2: "gelu"}[act]
    want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), name, torch.float32).numpy()
    scale = max(1.0, float(np.abs(want).max()))
    assert Hn.max_abs(d_y32.numpy(), want) <= 2e-4 * scale  # accumulation order only
    assert Hn.max_abs(d_y.numpy(), want) <= 1.5e-3 * scale  # one binary16 rounding of the result on top
    a, b = d_y32.numpy().astype(np.float16), d_y.numpy()
    if act != 2:
        assert np.array_equal(a, b)
    else:  # the two instantiations of the tanh-GELU epilogue may differ in the last binary32 bit
        ulp = np.spacing(np.maximum(np.abs(a), np.abs(b)).astype(np.float16)).astype(np.float32)
        assert np.all(np.abs(a.astype(np.float32) - b.astype(np.float32)) <= ulp)


@pytest.mark.parametrize("inp,out,sp", [(256, 128, 0.0), (768, 3072, 0.3), (3072, 768, 0.5), (64, 16, 0.9)])
def test_bsr16_dense_image(et, inp, out, sp):
    """The dense image the class multiplies with for weights that keep most of their tiles."""
    w = Hn.BsrWeight(out, inp, sp, seed=71)
    d_w = et.DeviceBuffer.empty((out, inp), np.float16)
    et.check(et.lib().et_fill_f16(d_w.ptr, out * inp, 0x7E00, None))
    et.check(et.lib().et_bsr16_to_dense_f16(up(et, w.row_ptr).ptr, up(et, w.col_idx).ptr, up(et, w.tiles).ptr, d_w.ptr,
                                            inp, out, None))
    want = F.bsr16_to_dense(w.row_ptr, w.col_idx, w.tiles, inp).astype(np.float16)
    assert np.array_equal(d_w.numpy(), want)


@pytest.mark.parametrize("T,inp,out,sp,act", [(1024, 768, 768, 0.8, 0), (1024, 3072, 768, 0.8, 0), (2048, 4096, 1024, 0.9, 0),
                                              (48, 64, 32, 0.3, 2), (64, 6144, 64, 0.5, 1), (4096, 768, 3072, 0.8, 2)])
def test_linear_bsr16_f32_output(et, T, inp, out, sp, act):
    """The binary32 store of the accumulator (mixed-precision residual stream): no rounding of
    the result, so the bound is accumulation-order noise only; and rounding it gives the
    binary16 entry point's result bit for bit."""
    w = Hn.BsrWeight(out, inp, sp, seed=21, bias_std=0.1).upload(et)
    x = Hn.randn((T, inp), 22)
    d_x = up(et, x)
    d_y32 = et.DeviceBuffer.empty((T, out), np.float32)
    d_y16 = et.DeviceBuffer.empty((T, out), np.float16)
    et.check(et.lib().et_linear_bsr16_f16_f32out(w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, w.d_bias.ptr,
                                                 d_x.ptr, d_y32.ptr, T, inp, out, act, None))
    w.forward(et, d_x, d_y16, T, act)
    want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), {0: None, 1: "relu", 2: "gelu"}[act], None).numpy()
    got = d_y32.numpy()
    assert Hn.max_abs(got, want) <= 5e-5 * max(1.0, float(np.abs(want).max()))
    a, b = got.astype(np.float16), d_y16.numpy()
    if act != 2:
        assert np.array_equal(a, b)
    else:
        # tanh-GELU is evaluated by two instantiations of the epilogue, whose fused multiply-adds
        # the compiler may contract differently: the last binary32 bit, hence rarely the binary16
        # rounding, can differ — by one unit in the last place at most
        ulp = np.spacing(np.maximum(np.abs(a), np.abs(b)).astype(np.float16)).astype(np.float32)
        assert np.all(np.abs(a.astype(np.float32) - b.astype(np.float32)) <= ulp)
        assert np.mean(a != b) < 1e-3


# Strips of 32 rows staged a half of the columns at a time: the smallest and the largest width, an odd number of column tiles, a last
# strip of 16 rows, one block-row a wave to four and waves with fewer, block-rows without tiles, with tiles in one
# half only, with all of them, and (ids drawn twice) with more tiles than columns; columns in any order.  "crowded": rows of no more tiles
# than columns, but more in one half than it has columns, in turn with ordinary rows of the same wave.
@pytest.mark.parametrize("T,inp,out,act", [(2048, 1280, 768, 0), (2064, 3072, 816, 2), (2064, 2000, 800, 1), (8208, 3056, 208, 0),
                                           (8192, 4096, 400, 0), (16400, 1296, 800, 2)])
@pytest.mark.parametrize("order", ["rising", "falling", "drawn", "twice", "crowded"])
def test_linear_bsr16_strip_halves(et, T, inp, out, act, order):
    rng = np.random.default_rng(inp + out)
    nc, rows = inp // 16, []
    for b in range(out // 16):
        lo, hi = ((0, nc), (0, nc), (0, (nc + 1) // 2), ((nc + 1) // 2, nc), (0, nc))[b % 5]
        n = (0, 1, 2, 15, 16, 17, 33, 64, 65, 1000)[int(rng.integers(0, 10))]
        ids = rng.permutation(np.arange(lo, hi))[:n]
        if order == "twice" and b % 3 == 0:
            ids = rng.integers(0, nc, nc + 1 + int(rng.integers(0, 70)))
        if order == "crowded" and (b // 12 + b) % 2 == 0:
            lo, hi = ((0, (nc + 1) // 2), ((nc + 1) // 2, nc))[b // 2 % 2]
            ids = rng.integers(lo, hi, int(rng.integers((nc + 1) // 2 + 1, nc + 1)))
        rows.append({"rising": np.sort(ids), "falling": -np.sort(-ids)}.get(order, ids))
    row_ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col_idx = np.concatenate(rows).astype(np.int32)
    tiles, bias, x = Hn.randn((len(col_idx), 256), 1, 0.02), Hn.randn((out,), 2, 0.1), Hn.randn((T, inp), 3)
    dense = np.zeros((out, inp), np.float32)
    for b in range(out // 16):
        for t in range(row_ptr[b], row_ptr[b + 1]):
            dense[16 * b:16 * b + 16, 16 * col_idx[t]:16 * col_idx[t] + 16] += tiles[t].reshape(16, 16).astype(np.float32)
    d = [up(et, v) for v in (row_ptr, col_idx, tiles, bias, x)]
    d_y, d_y32 = up(et, np.full((T + 16, out), 7, np.float16)), up(et, np.full((T + 16, out), 7, np.float32))
    et.check(et.lib().et_linear_bsr16_f16(*[v.ptr for v in d], d_y.ptr, T, inp, out, act, None))
    et.check(et.lib().et_linear_bsr16_f16_f32out(*[v.ptr for v in d], d_y32.ptr, T, inp, out, act, None))
    want = L.linear(Hn.f32(x), Hn.f32(dense), Hn.f32(bias), {0: None, 1: "relu", 2: "gelu"}[act], None).numpy()
    scale = max(1.0, float(np.abs(want).max()))
    y, y32 = d_y.numpy(), d_y32.numpy()
    # binary32 sums of at most 2 x 4096 exact products (a column drawn twice is one sum in the reference): order of
    # accumulation only; a binary16 rounding of the result on top
    assert Hn.max_abs(y32[:T], want) <= 5e-5 * scale
    assert Hn.max_abs(y[:T], want) <= 1e-3 * scale
    assert (y[T:] == 7).all() and (y32[T:] == 7).all()


# The call that knows the number of tiles, on both sides of its line between strips of 16 rows and strips in halves (an estimate of
# either: few tiles; one workgroup a compute unit and more; rows a workgroup deals unevenly), and with a count that is not known.
@pytest.mark.parametrize("T,inp,out", [(2048, 3072, 768), (4096, 3072, 768), (3072, 4096, 1024), (2064, 1536, 1536), (8192, 2048, 208)])
@pytest.mark.parametrize("sp", [0.8, 0.95, 1.0])
@pytest.mark.parametrize("act", [0, 2])
def test_linear_bsr16_counted(et, T, inp, out, sp, act):
    w = Hn.BsrWeight(out, inp, sp, seed=inp + out, std=0.02, bias_std=0.1)
    n = len(w.col_idx)
    x = Hn.randn((T, inp), 3)
    want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), {0: None, 2: "gelu"}[act], None).numpy()
    d = [up(et, v if len(v) else np.zeros(256, v.dtype)) for v in (w.row_ptr, w.col_idx, w.tiles)]
    d_b, d_x = up(et, w.bias), up(et, x)
    for count in (n, -1):
        d_y, d_y32 = up(et, np.full((T + 16, out), 7, np.float16)), up(et, np.full((T + 16, out), 7, np.float32))
        et.check(et.lib().et_linear_bsr16_counted_f16(*[v.ptr for v in d], count, d_b.ptr, d_x.ptr, d_y.ptr, T, inp, out, act, None))
        et.check(et.lib().et_linear_bsr16_counted_f16_f32out(*[v.ptr for v in d], count, d_b.ptr, d_x.ptr, d_y32.ptr, T, inp, out, act, None))
        y, y32 = d_y.numpy(), d_y32.numpy()
        # as for the strips in halves: order of accumulation, and a binary16 rounding of the result on top
        assert Hn.max_abs(y32[:T], want) <= 5e-5 and Hn.max_abs(y[:T], want) <= 1e-3 * max(1.0, float(np.abs(want).max()))
        assert (y[T:] == 7).all() and (y32[T:] == 7).all()


PLANNED_CASES = [
    # T, in, out, sparsity, act, (mt, kc, rows_per_wg) or None for the automatic geometry
    (1024, 768, 2304, 0.8, 0, None),
    (1024, 768, 768, 0.8, 0, None),
    (1024, 768, 3072, 0.8, 2, None),
    (1024, 3072, 768, 0.8, 0, None),
    (2048, 4096, 1024, 0.9, 0, None),
    (2048, 768, 3072, 0.9, 1, None),
    (8192, 768, 768, 0.8, 2, None),       # 128-row strips
    (128, 800, 208, 0.5, 1, None),        # widths that are no multiple of the chunk, 13 block-rows
    (64, 6144, 64, 0.5, 0, None),         # an input no LDS strip of the plain kernel holds
    (1040, 768, 768, 0.8, 1, None),       # ragged last strip
    (16, 128, 16, 0.0, 0, None),
    (48, 256, 32, 0.3, 2, (1, 128, 1)),
    (2048, 768, 3072, 0.0, 0, (4, 128, 12)),   # dense structure, two block-rows per wave in half of the waves
    (512, 3072, 768, 0.8, 0, (2, 512, 3)),
    (512, 3072, 768, 0.8, 0, (8, 128, 24)),
    (256, 1024, 1024, 0.95, 0, (1, 512, 20)),  # block-rows without tiles in most chunks
    (64, 8320, 64, 0.5, 0, (1, 128, 4)),       # 65 chunks: the per-chunk tables are reloaded after 64
    (32, 16512, 32, 0.8, 1, (1, 128, 2)),      # 129 chunks
]


@pytest.mark.parametrize("T,inp,out,sp,act,geom", PLANNED_CASES)
def test_linear_bsr16_planned(et, T, inp, out, sp, act, geom):
    """The streaming kernel behind a plan: same Linear as the plain call, for binary16 and
    binary32 results, at the automatic and at forced launch geometries."""
    import ctypes as C
    lib = et.lib()
    w = Hn.BsrWeight(out, inp, sp, seed=31, bias_std=0.1).upload(et)
    x = Hn.randn((T, inp), 32)
    d_x = up(et, x)
    mt, kc, rpw = geom or (0, 0, 0)
    plan = C.c_void_p()
    et.check(lib.et_bsr16_plan_create(w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, T, inp, out, mt, kc, rpw,
                                      C.byref(plan)))
    try:
        g = [C.c_int() for _ in range(4)]
        et.check(lib.et_bsr16_plan_info(plan, *[C.byref(v) for v in g]))
        d_y16 = et.DeviceBuffer.empty((T, out), np.float16)
        d_y32 = et.DeviceBuffer.empty((T, out), np.float32)
        et.check(lib.et_fill_f16(d_y16.ptr, T * out, 0x7E00, None))
        et.check(lib.et_linear_bsr16_planned_f16(plan, w.d_bias.ptr, d_x.ptr, d_y16.ptr, None, T, act, None))
        et.check(lib.et_linear_bsr16_planned_f16(plan, w.d_bias.ptr, d_x.ptr, None, d_y32.ptr, T, act, None))
        name = {0: None, 1: "relu", 2: "gelu"}[act]
        want32 = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), name, None).numpy()
        want16 = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), name, torch.float16).numpy()
        e16, e32 = Hn.max_abs(d_y16.numpy(), want16), Hn.max_abs(d_y32.numpy(), want32)
        print(f"planned T={T} in={inp} out={out} sp={sp} geometry mt={g[0].value} kc={g[1].value} rows={g[2].value} "
              f"lds={g[3].value}: max-abs fp16 {e16:.2e} fp32 {e32:.2e}")
        assert e16 <= 4e-3
        assert e32 <= 5e-5 * max(1.0, float(np.abs(want32).max()))
        # a plan serves other row counts too (here: the first 16 rows only)
        d_y = et.DeviceBuffer.empty((16, out), np.float16)
        et.check(lib.et_linear_bsr16_planned_f16(plan, w.d_bias.ptr, d_x.ptr, d_y.ptr, None, 16, act, None))
        assert Hn.max_abs(d_y.numpy(), want16[:16]) <= 4e-3
    finally:
        et.check(lib.et_bsr16_plan_destroy(plan))


def test_bsr16_plan_rejects_what_it_cannot_do(et):
    import ctypes as C
    lib = et.lib()
    w = Hn.BsrWeight(64, 64, 0.5, seed=33).upload(et)
    plan = C.c_void_p()
    args = (w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr)
    assert lib.et_bsr16_plan_create(*args, 64, 64, 64, 0, 0, 0, C.byref(plan)) == et.ET_ERR_UNSUPPORTED  # in < 128
    assert lib.et_bsr16_plan_create(*args, 64, 64, 64, 3, 0, 0, C.byref(plan)) != et.ET_OK
    w2 = Hn.BsrWeight(512, 2048, 0.0, seed=34).upload(et)
    # 32 dense block-rows of 512 columns per chunk: 512 slots = 512 KB of LDS per buffer
    st = lib.et_bsr16_plan_create(w2.d_row_ptr.ptr, w2.d_col_idx.ptr, w2.d_tiles.ptr, 64, 2048, 512, 1, 512, 32,
                                  C.byref(plan))
    assert st == et.ET_ERR_UNSUPPORTED and b"LDS" in lib.et_last_error()
    assert plan.value is None


def test_linear_bsr16_closed_form_all_ones(et):
    """All-ones input and all-ones tiles: Y[t][o] = 16 * tiles_in_block_row(o/16) + bias
    (the only closed form the reference's driver offers, Linear/test/test_tile.cu:56-75)."""
    T, inp, out = 64, 256, 128
    row_ptr, col_idx = F.gen_tile_pattern(out, inp, 0.6, seed=5)
    tiles = np.ones((len(col_idx), 256), np.float16)
    bias = np.full(out, 0.5, np.float16)
    x = np.ones((T, inp), np.float16)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    et.linear_bsr16(up(et, row_ptr), up(et, col_idx), up(et, tiles), up(et, bias), up(et, x), d_y, T, inp, out)
    per_row = np.diff(row_ptr)
    want = np.repeat(16.0 * per_row + 0.5, 16)[None, :].repeat(T, 0)
    assert np.array_equal(d_y.numpy().astype(np.float32), want.astype(np.float32))


def test_linear_bsr16_empty_rows_and_no_bias(et):
    T, inp, out = 32, 64, 64
    row_ptr = np.array([0, 0, 2, 2, 3], np.int32)  # block-rows 0 and 2 hold no tile
    col_idx = np.array([3, 0, 1], np.int32)
    tiles = Hn.randn((3, 256), 21, 0.5)
    x = Hn.randn((T, inp), 22)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    et.check(et.lib().et_fill_f16(d_y.ptr, T * out, 0x7E00, None))  # NaN: every element must be written
    et.linear_bsr16(up(et, row_ptr), up(et, col_idx), up(et, tiles), None, up(et, x), d_y, T, inp, out)
    W = F.bsr16_to_dense(row_ptr, col_idx, tiles, inp)
    want = L.linear(Hn.f32(x), Hn.f32(W), None, None, torch.float16).numpy()
    got = d_y.numpy()
    assert np.all(got[:, :16] == 0) and np.all(got[:, 32:48] == 0)
    assert Hn.max_abs(got, want) <= 4e-3


def test_linear_bsr16_tile_order_is_free(et):
    """Permuting the tiles inside each block-row (with their column ids) leaves Y unchanged
    up to accumulation order."""
    T, inp, out = 64, 256, 64
    w = Hn.BsrWeight(out, inp, 0.5, seed=31)
    col2, tiles2 = w.col_idx.copy(), w.tiles.copy()
    for r in range(out // 16):
        lo, hi = w.row_ptr[r], w.row_ptr[r + 1]
        col2[lo:hi] = w.col_idx[lo:hi][::-1]
        tiles2[lo:hi] = w.tiles[lo:hi][::-1]
    x = Hn.randn((T, inp), 32)
    d_x = up(et, x)
    ys = []
    for c, t in ((w.col_idx, w.tiles), (col2, tiles2)):
        d_y = et.DeviceBuffer.empty((T, out), np.float16)
        et.linear_bsr16(up(et, w.row_ptr), up(et, c), up(et, t), None, d_x, d_y, T, inp, out)
        ys.append(d_y.numpy())
    assert Hn.max_abs(ys[0], ys[1]) <= 1e-3


def test_linear_bsr16_rejects_bad_args(et):
    d = et.DeviceBuffer.empty((64, 64), np.float16)
    f = et.lib().et_linear_bsr16_f16
    assert f(d.ptr, d.ptr, d.ptr, None, d.ptr, d.ptr, 20, 64, 64, 0, None) == et.ET_ERR_UNSUPPORTED
    assert f(None, d.ptr, d.ptr, None, d.ptr, d.ptr, 16, 64, 64, 0, None) == et.ET_ERR_INVALID_ARG
    assert f(d.ptr, d.ptr, d.ptr, None, d.ptr, d.ptr, 16, 64, 64, 9, None) == et.ET_ERR_INVALID_ARG
    assert f(d.ptr, d.ptr, d.ptr, None, d.ptr, d.ptr, 0, 64, 64, 0, None) == et.ET_OK  # empty batch


@pytest.mark.parametrize("T,inp,out,sp,act", [(1024, 768, 3072, 0.8, 2), (1008, 768, 3072, 0.8, 2),
                                               (48, 256, 512, 0.5, 1), (16, 1024, 256, 0.9, 0),
                                               (64, 2048, 256, 0.9, 0), (128, 72 * 4, 160, 0.6, 2)])
def test_skipln_linear_bsr16(et, T, inp, out, sp, act):
    """SkipLayerNorm fused into the tile-sparse Linear: same values as the two operators
    launched one after the other (in > 1024 takes that route inside the call)."""
    if inp % 16:
        pytest.skip("feature width must be a multiple of 16")
    w = Hn.BsrWeight(out, inp, sp, seed=21, bias_std=0.05).upload(et)
    src, skip = Hn.randn((T, inp), 22), Hn.randn((T, inp), 23)
    gamma = (1 + Hn.randn((inp,), 24, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((inp,), 25, 0.1)
    d_src, d_skip, d_g, d_b = up(et, src), up(et, skip), up(et, gamma), up(et, beta)
    d_ln = et.DeviceBuffer.empty((T, inp), np.float16)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    et.check(et.lib().et_skipln_linear_bsr16_f16(d_src.ptr, d_skip.ptr, d_g.ptr, d_b.ptr, 1e-5, d_ln.ptr,
                                                 w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, w.d_bias.ptr,
                                                 d_y.ptr, T, inp, out, act, None))
    et.sync()
    # the two separate operators
    d_ln2 = et.DeviceBuffer.empty((T, inp), np.float16)
    d_y2 = et.DeviceBuffer.empty((T, out), np.float16)
    et.skip_layernorm(d_ln2, d_src, d_skip, d_g, d_b, T, inp, 1e-5)
    w.forward(et, d_ln2, d_y2, T, act)
    et.sync()
    ln, ln2 = d_ln.numpy(), d_ln2.numpy()
    # the normalised rows may differ by one fp16 rounding where fp32 contraction differs
    assert Hn.max_abs(ln, ln2) <= 4e-3
    want_ln = L.skip_layernorm(Hn.f32(src), Hn.f32(skip), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    assert Hn.max_abs(ln, want_ln.numpy()) <= 4e-3
    # the Linear consumes exactly the rows it wrote: oracle on ln_out
    want = L.linear(Hn.f32(ln), Hn.f32(w.dense), Hn.f32(w.bias), {0: None, 1: "relu", 2: "gelu"}[act],
                    torch.float16)
    assert Hn.max_abs(d_y.numpy(), want.numpy()) <= 5e-3
    assert Hn.max_abs(d_y.numpy(), d_y2.numpy()) <= 2e-2


def test_skipln_linear_bsr16_in_place_falls_back(et):
    """ln_out aliasing src is legal: the call then runs the two operators back to back."""
    T, inp, out = 64, 256, 256
    w = Hn.BsrWeight(out, inp, 0.5, seed=31, bias_std=0.05).upload(et)
    src, skip = Hn.randn((T, inp), 32), Hn.randn((T, inp), 33)
    gamma, beta = np.ones(inp, np.float16), np.zeros(inp, np.float16)
    d_src, d_skip, d_g, d_b = up(et, src), up(et, skip), up(et, gamma), up(et, beta)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    et.check(et.lib().et_skipln_linear_bsr16_f16(d_src.ptr, d_skip.ptr, d_g.ptr, d_b.ptr, 1e-5, d_src.ptr,
                                                 w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, w.d_bias.ptr,
                                                 d_y.ptr, T, inp, out, 0, None))
    et.sync()
    want_ln = L.skip_layernorm(Hn.f32(src), Hn.f32(skip), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16)
    assert Hn.max_abs(d_src.numpy(), want_ln.numpy()) <= 4e-3
    want = L.linear(Hn.f32(d_src.numpy()), Hn.f32(w.dense), Hn.f32(w.bias), None, torch.float16)
    assert Hn.max_abs(d_y.numpy(), want.numpy()) <= 5e-3


@pytest.mark.parametrize("T,n_in,n_mid,n_out,sp,act", [(1024, 768, 768, 3072, 0.8, 2), (1024, 3072, 768, 2304, 0.8, 0),
                                                     (48, 256, 512, 64, 0.5, 1), (16, 32, 16, 16, 0.0, 0),
                                                     (2048, 4096, 1024, 4096, 0.9, 2), (272, 160, 208, 800, 0.5, 0)])
def test_split_layernorm_between_two_tile_linears(et, T, n_in, n_mid, n_out, sp, act):
    """Producer Linear (row statistics of output + residual) -> consumer Linear (adds the two and
    normalises while staging): V, the statistics, the normalised rows and Y against the oracle;
    the stand-alone normalisation from the same statistics is bit-identical to the fused one."""
    import ctypes as C
    lib = et.lib()
    w1 = Hn.BsrWeight(n_mid, n_in, sp, seed=41, bias_std=0.05).upload(et)
    w2 = Hn.BsrWeight(n_out, n_mid, sp, seed=44, bias_std=0.05).upload(et)
    x, resid = Hn.randn((T, n_in), 47), Hn.randn((T, n_mid), 48)
    gamma = (1 + Hn.randn((n_mid,), 49, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((n_mid,), 50, 0.1)
    d_v = et.DeviceBuffer.empty((T, n_mid), np.float16)
    d_stats = et.DeviceBuffer.empty((16, T, 2), np.float32)
    d_resid = up(et, resid)
    groups = C.c_int(0)
    assert lib.et_linear_bsr16_fused_ln_supported(T, n_in, n_mid) == 1
    et.check(lib.et_linear_bsr16_resid_stats_f16(w1.d_row_ptr.ptr, w1.d_col_idx.ptr, w1.d_tiles.ptr, w1.d_bias.ptr,
                                                 up(et, x).ptr, d_resid.ptr, d_v.ptr, d_stats.ptr,
                                                 C.byref(groups), T, n_in, n_mid, None))
    G = groups.value
    assert 1 <= G <= 16
    v = d_v.numpy()
    want_v = L.linear(Hn.f32(x), Hn.f32(w1.dense), Hn.f32(w1.bias), None, torch.float16).numpy()
    assert Hn.max_abs(v, want_v) <= 4e-3  # the plain Linear output
    st = d_stats.numpy()[:G].astype(np.float64).sum(0)
    s64 = v.astype(np.float64) + resid.astype(np.float64)
    assert np.allclose(st[:, 0], s64.sum(1), rtol=1e-5, atol=1e-3)
    assert np.allclose(st[:, 1], (s64 * s64).sum(1), rtol=1e-5, atol=1e-3)

    d_ln = et.DeviceBuffer.empty((T, n_mid), np.float16)
    d_y = et.DeviceBuffer.empty((T, n_out), np.float16)
    d_g, d_b = up(et, gamma), up(et, beta)
    et.check(lib.et_norm_linear_bsr16_f16(d_v.ptr, d_resid.ptr, d_stats.ptr, G, d_g.ptr, d_b.ptr, 1e-5, d_ln.ptr,
                                          w2.d_row_ptr.ptr, w2.d_col_idx.ptr, w2.d_tiles.ptr, w2.d_bias.ptr, d_y.ptr,
                                          T, n_mid, n_out, act, None))
    ln = d_ln.numpy()
    want_ln = L.skip_layernorm(Hn.f32(v), Hn.f32(resid), Hn.f32(gamma), Hn.f32(beta), 1e-5, torch.float16).numpy()
    assert Hn.max_abs(ln, want_ln) <= 4e-3
    want_y = L.linear(Hn.f32(ln), Hn.f32(w2.dense), Hn.f32(w2.bias), {0: None, 1: "relu", 2: "gelu"}[act],
                      torch.float16).numpy()
    assert Hn.max_abs(d_y.numpy(), want_y) <= 5e-3

    d_ln2 = et.DeviceBuffer.empty((T, n_mid), np.float16)
    et.check(lib.et_norm_from_stats_f16(d_ln2.ptr, d_v.ptr, d_resid.ptr, d_stats.ptr, G, d_g.ptr, d_b.ptr, T, n_mid,
                                        1e-5, None))
    assert np.array_equal(d_ln2.numpy().view(np.uint16), ln.view(np.uint16))


def _random_split_cases(n, seed):
    rng = np.random.default_rng(seed)
    return [(16 * int(rng.integers(1, 21)), 16 * int(rng.integers(1, 49)), 16 * int(rng.integers(1, 129)),
             16 * int(rng.integers(1, 65)), float(rng.choice([0.0, 0.5, 0.8, 0.9, 0.97])), int(rng.integers(0, 3)))
            for _ in range(n)]


@pytest.mark.parametrize("T,n_in,n_mid,n_out,sp,act", [(1024, 768, 768, 3072, 0.8, 2), (1024, 3072, 768, 2304, 0.8, 0),
                                                     (48, 256, 512, 64, 0.5, 1), (16, 32, 16, 16, 0.0, 0),
                                                     (2048, 4096, 1024, 4096, 0.9, 2), (272, 160, 208, 800, 0.5, 0),
                                                     (48, 256, 4224, 64, 0.5, 0)]  # rows wider than two passes of 256 threads
                         + _random_split_cases(16, 20211115))
def test_split_layernorm_binary32_between_two_tile_linears(et, T, n_in, n_mid, n_out, sp, act):
    """The split normalisation of the mixed-precision layer: the producer stores X W^T + b + residual
    unrounded with its row sums, the consumer normalises that strip while staging it and writes
    the normalised rows as binary32 and binary16."""
    import ctypes as C
    lib = et.lib()
    w1 = Hn.BsrWeight(n_mid, n_in, sp, seed=41, bias_std=0.05).upload(et)
    w2 = Hn.BsrWeight(n_out, n_mid, sp, seed=44, bias_std=0.05).upload(et)
    x = Hn.randn((T, n_in), 47)
    resid = Hn.randn((T, n_mid), 48, 1.0, np.float32)
    gamma = (1 + Hn.randn((n_mid,), 49, 0.1, np.float32)).astype(np.float16)
    beta = Hn.randn((n_mid,), 50, 0.1)
    d_v = et.DeviceBuffer.empty((T, n_mid), np.float32)
    d_stats = et.DeviceBuffer.empty((16, T, 2), np.float32)
    groups = C.c_int(0)
    assert lib.et_linear_bsr16_resid_stats_f32_supported(T, n_in, n_mid) == 1
    assert lib.et_norm_linear_bsr16_f32in_supported(T, n_mid, n_out) == 1
    et.check(lib.et_linear_bsr16_resid_stats_f32(w1.d_row_ptr.ptr, w1.d_col_idx.ptr, w1.d_tiles.ptr, w1.d_bias.ptr,
                                                 up(et, x).ptr, up(et, resid).ptr, None, None, None, d_v.ptr,
                                                 d_stats.ptr, C.byref(groups), T, n_in, n_mid, None))
    G = groups.value
    assert 1 <= G <= 16
    v = d_v.numpy()
    want_v = L.linear(Hn.f32(x), Hn.f32(w1.dense), Hn.f32(w1.bias)).numpy() + resid
    assert Hn.max_abs(v, want_v) <= 1e-4 * max(1.0, float(np.abs(want_v).max()))
    st = d_stats.numpy()[:G].astype(np.float64).sum(0)
    v64 = v.astype(np.float64)
    assert np.allclose(st[:, 0], v64.sum(1), rtol=1e-5, atol=1e-3)
    assert np.allclose(st[:, 1], (v64 * v64).sum(1), rtol=1e-5, atol=1e-3)

    d_ln32 = et.DeviceBuffer.empty((T, n_mid), np.float32)
    d_ln16 = et.DeviceBuffer.empty((T, n_mid), np.float16)
    d_y = et.DeviceBuffer.empty((T, n_out), np.float16)
    et.check(lib.et_fill_f16(d_ln16.ptr, T * n_mid, 0x7E00, None))
    d_g, d_b = up(et, gamma), up(et, beta)
    d_fin = et.DeviceBuffer.empty((T, 2), np.float32)
    et.check(lib.et_norm_linear_bsr16_f32in(d_v.ptr, d_stats.ptr, G, d_g.ptr, d_b.ptr, 1e-5, d_fin.ptr, d_ln32.ptr, d_ln16.ptr,
                                            w2.d_row_ptr.ptr, w2.d_col_idx.ptr, w2.d_tiles.ptr, w2.d_bias.ptr, d_y.ptr,
                                            T, n_mid, n_out, act, None))
    ln32, ln16 = d_ln32.numpy(), d_ln16.numpy()
    fin = d_fin.numpy().astype(np.float64)
    assert np.allclose(fin[:, 0], v64.mean(1), rtol=1e-5, atol=1e-5)
    assert np.allclose(fin[:, 1], 1 / np.sqrt(v64.var(1) + 1e-5), rtol=1e-4)
    want_ln = L.layernorm(torch.from_numpy(v), Hn.f32(gamma), Hn.f32(beta), 1e-5).numpy()
    assert Hn.max_abs(ln32, want_ln) <= 2e-4 * max(1.0, float(np.abs(want_ln).max()))
    assert np.array_equal(ln16.view(np.uint16), ln32.astype(np.float16).view(np.uint16))  # one value, two roundings
    want_y = L.linear(Hn.f32(ln16), Hn.f32(w2.dense), Hn.f32(w2.bias), {0: None, 1: "relu", 2: "gelu"}[act],
                      torch.float16).numpy()
    assert Hn.max_abs(d_y.numpy(), want_y) <= 5e-3
    # without the binary16 copy (what the layer asks for) Y does not change
    d_y2 = et.DeviceBuffer.empty((T, n_out), np.float16)
    et.check(lib.et_norm_linear_bsr16_f32in(d_v.ptr, d_stats.ptr, G, d_g.ptr, d_b.ptr, 1e-5, None, d_ln32.ptr, None,
                                            w2.d_row_ptr.ptr, w2.d_col_idx.ptr, w2.d_tiles.ptr, w2.d_bias.ptr, d_y2.ptr,
                                            T, n_mid, n_out, act, None))
    assert np.array_equal(d_y2.numpy().view(np.uint16), d_y.numpy().view(np.uint16))
    # the stand-alone normalisation from the same sums is bit-identical
    d_o32 = et.DeviceBuffer.empty((T, n_mid), np.float32)
    d_o16 = et.DeviceBuffer.empty((T, n_mid), np.float16)
    et.check(lib.et_norm_from_stats_f32in(d_o32.ptr, d_o16.ptr, d_v.ptr, d_stats.ptr, G, d_g.ptr, d_b.ptr, T, n_mid,
                                          1e-5, None))
    assert np.array_equal(d_o32.numpy().view(np.uint32), ln32.view(np.uint32))
    assert np.array_equal(d_o16.numpy().view(np.uint16), ln16.view(np.uint16))
    # a second producer whose residual is that normalisation, formed in its epilogue from V and the sums
    # instead of being read: the same result as with the stored rows
    w3 = Hn.BsrWeight(n_mid, n_out, sp, seed=45, bias_std=0.05).upload(et)
    d_v2a, d_v2b = et.DeviceBuffer.empty((T, n_mid), np.float32), et.DeviceBuffer.empty((T, n_mid), np.float32)
    d_st2a, d_st2b = et.DeviceBuffer.empty((16, T, 2), np.float32), et.DeviceBuffer.empty((16, T, 2), np.float32)
    g2 = C.c_int(0)
    common = (w3.d_row_ptr.ptr, w3.d_col_idx.ptr, w3.d_tiles.ptr, w3.d_bias.ptr, d_y.ptr)
    et.check(lib.et_linear_bsr16_resid_stats_f32(*common, d_ln32.ptr, None, None, None, d_v2a.ptr, d_st2a.ptr,
                                                 C.byref(g2), T, n_out, n_mid, None))
    et.check(lib.et_linear_bsr16_resid_stats_f32(*common, d_v.ptr, d_fin.ptr, d_g.ptr, d_b.ptr, d_v2b.ptr,
                                                 d_st2b.ptr, C.byref(g2), T, n_out, n_mid, None))
    assert np.array_equal(d_v2a.numpy().view(np.uint32), d_v2b.numpy().view(np.uint32))
    # a binary16 residual (the first layer of a stack adds the model's input): the same bits as with its widened copy
    r16 = Hn.randn((T, n_mid), 46)
    d_v2c, d_v2d = et.DeviceBuffer.empty((T, n_mid), np.float32), et.DeviceBuffer.empty((T, n_mid), np.float32)
    d_st2c, d_st2d = et.DeviceBuffer.empty((16, T, 2), np.float32), et.DeviceBuffer.empty((16, T, 2), np.float32)
    et.check(lib.et_linear_bsr16_resid_stats_f32(*common, et.DeviceBuffer.from_numpy(r16.astype(np.float32)).ptr, None, None,
                                                 None, d_v2c.ptr, d_st2c.ptr, C.byref(g2), T, n_out, n_mid, None))
    et.check(lib.et_linear_bsr16_resid16_stats_f32(*common, et.DeviceBuffer.from_numpy(r16).ptr, d_v2d.ptr, d_st2d.ptr,
                                                   C.byref(g2), T, n_out, n_mid, None))
    assert np.array_equal(d_v2c.numpy().view(np.uint32), d_v2d.numpy().view(np.uint32))
    # (its row sums are added over 8 waves where the binary32 form may run 12: the same numbers up to the order)
    assert np.allclose(d_st2c.numpy()[: g2.value], d_st2d.numpy()[: g2.value], rtol=2e-6, atol=1e-4)
    assert np.array_equal(d_st2a.numpy()[:g2.value].view(np.uint32), d_st2b.numpy()[:g2.value].view(np.uint32))
    want_v2 = L.linear(Hn.f32(d_y.numpy()), Hn.f32(w3.dense), Hn.f32(w3.bias)).numpy() + want_ln
    assert Hn.max_abs(d_v2b.numpy(), want_v2) <= 3e-4 * max(1.0, float(np.abs(want_v2).max()))



def test_split_layernorm_rejects_unsupported(et):
    import ctypes as C
    lib = et.lib()
    assert lib.et_linear_bsr16_fused_ln_supported(64, 6144, 64) == 0  # strip does not fit in LDS
    assert lib.et_linear_bsr16_fused_ln_supported(64, 60, 64) == 0
    d = et.DeviceBuffer.empty((64, 64), np.float16)
    g = C.c_int(0)
    st = lib.et_norm_linear_bsr16_f16(d.ptr, d.ptr, d.ptr, 17, d.ptr, d.ptr, 1e-5, d.ptr, d.ptr, d.ptr, d.ptr, d.ptr,
                                      d.ptr, 64, 64, 64, 0, None)
    assert st == et.ET_ERR_INVALID_ARG


@pytest.mark.parametrize("mt,stage,threads,rpw", [(1, 1, 256, 4), (2, 1, 128, 3), (4, 1, 512, 8),
                                                  (4, 0, 256, 5), (1, 0, 64, 1), (2, 0, 512, 48),
                                                  (1, 1, 768, 24), (2, 1, 768, 48), (1, 1, 640, 7), (2, 1, 576, 10)])  # the 12-wave form
def test_linear_bsr16_every_geometry(et, mt, stage, threads, rpw):
    """Each launch geometry of the kernel gives the same result, including a token count that
    is not a multiple of the strip."""
    T, inp, out = 80, 768, 768
    w = Hn.BsrWeight(out, inp, 0.8, seed=41, bias_std=0.1).upload(et)
    x = Hn.randn((T, inp), 42)
    d_y = et.DeviceBuffer.empty((T, out), np.float16)
    et.check(et.lib().et_linear_bsr16_f16_geom(w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr, w.d_bias.ptr,
                                               up(et, x).ptr, d_y.ptr, T, inp, out, 2, mt, stage, threads, rpw,
                                               None))
    want = L.linear(Hn.f32(x), Hn.f32(w.dense), Hn.f32(w.bias), "gelu", torch.float16)
    assert Hn.max_abs(d_y.numpy(), want.numpy()) <= 4e-3


def test_linear_bsr16_geometry_limits(et):
    """64-row strips have no 12-wave form, and no geometry runs more than 12 waves: refused, not launched."""
    w = Hn.BsrWeight(768, 768, 0.8, seed=41).upload(et)
    d = et.DeviceBuffer.empty((64, 768), np.float16)
    call = lambda mt, threads: et.lib().et_linear_bsr16_f16_geom(w.d_row_ptr.ptr, w.d_col_idx.ptr, w.d_tiles.ptr,
                                                               w.d_bias.ptr, d.ptr, d.ptr, 64, 768, 768, 0, mt, 1, threads,
                                                               8, None)
    assert call(4, 768) == et.ET_ERR_INVALID_ARG
    assert call(1, 832) == et.ET_ERR_INVALID_ARG


# ---------------------------------------------------------------- attention --

def run_mha(et, B, S, nh, hd, seed, lens=None, causal=False, mask=None, single_buffer=False, pad=0):
    """pad: halfs between the rows of the result, which keep what they held."""
    H = nh * hd
    T = B * S
    if single_buffer:
        qkv = Hn.randn((T, 3 * H), seed, 1.0)
        d_qkv = up(et, qkv)
        q, k, v = qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:]
        pq, pk, pv, ld = d_qkv.ptr, d_qkv.offset(2 * H), d_qkv.offset(4 * H), 3 * H
        keep = [d_qkv]
    else:
        q, k, v = Hn.randn((T, H), seed), Hn.randn((T, H), seed + 1), Hn.randn((T, H), seed + 2)
        keep = [up(et, q), up(et, k), up(et, v)]
        pq, pk, pv, ld = keep[0].ptr, keep[1].ptr, keep[2].ptr, H
    ldz = H + pad
    d_z = et.DeviceBuffer.empty((T, ldz), np.float16)
    et.check(et.lib().et_fill_f16(d_z.ptr, T * ldz, 0x7E00, None))
    d_lens = up(et, np.asarray(lens, np.int32)) if lens is not None else None
    d_mask = up(et, mask.astype(np.float16)) if mask is not None else None
    et.mha_fused(pq, pk, pv, ld, ld, ld, d_z, ldz, d_mask, d_lens, B, S, nh, hd, 1.0 / math.sqrt(hd),
                 et.MHA_CAUSAL if causal else 0)
    want = L.mha(Hn.f32(q), Hn.f32(k), Hn.f32(v), nh, B, mask=None if mask is None else Hn.f32(mask),
                 lens=lens, causal=causal, store=torch.float16)
    got = d_z.numpy()
    assert (got[:, H:].view(np.uint16) == 0x7E00).all()
    return np.ascontiguousarray(got[:, :H]), want.numpy()


@pytest.mark.parametrize("B", [1, 4, 16])
def test_attention_block_dense_projections_padded(et, B):
    """The fused self-attention block composed as a caller composes it: dense Q, K, V and O
    projections (768 x 768, N(0, 0.02)) around the fused attention core, S128, 12 heads x 64,
    inputs N(0,1), right padding with lengths in [64, 128] — against the oracle's attention block."""
    H, nh, S = 768, 12, 128
    T, hd = B * S, 64
    g = Hn.rng(300 + B)
    W = {k: (torch.randn(H, H, generator=g) * 0.02).numpy().astype(np.float16) for k in "qkvo"}
    x = Hn.randn((T, H), 310 + B)
    lens = torch.randint(64, 129, (B,), generator=Hn.rng(320 + B)).numpy().astype(np.int32)
    d_x, d_lens = up(et, x), up(et, lens)
    d = {k: et.DeviceBuffer.empty((T, H), np.float16) for k in ("q", "k", "v", "z", "out")}
    for k in "qkv":
        et.linear_dense(up(et, W[k]), None, d_x, d[k], T, H, H)
    et.mha_fused(d["q"], d["k"], d["v"], H, H, H, d["z"], H, None, d_lens, B, S, nh, hd, 1.0 / math.sqrt(hd))
    et.linear_dense(up(et, W["o"]), None, d["z"], d["out"], T, H, H)
    Wqkv = np.concatenate([W["q"], W["k"], W["v"]])
    zeros = torch.zeros
    P = L.LayerParams(Hn.f32(Wqkv), zeros(3 * H), Hn.f32(W["o"]), zeros(H), None, None, None, None, None, None, None, None)
    want16 = L.attention_block(Hn.f32(x), P, L.LayerConfig(nh=nh, B=B, lens=torch.as_tensor(lens), store=torch.float16))
    want32 = L.attention_block(Hn.f32(x), P, L.LayerConfig(nh=nh, B=B, lens=torch.as_tensor(lens), store=None))
    got = d["out"].numpy()
    e16, e32 = Hn.max_abs(got, want16.numpy()), Hn.max_abs(got, want32.numpy())
    print(f"attention block B={B} lens={lens.tolist()}: vs fp16-storage oracle {e16:.2e}, vs fp32 {e32:.2e}")
    assert e16 <= 2e-3 and e32 <= 2e-2
    # rows of padded queries are computed too (only keys are masked), and padding never leaks:
    # each sequence alone gives the same rows
    b = B - 1
    d1 = {k: et.DeviceBuffer.empty((S, H), np.float16) for k in ("z", "out")}
    off = b * S * H * 2
    et.mha_fused(d["q"].offset(off), d["k"].offset(off), d["v"].offset(off), H, H, H, d1["z"], H, None,
                 up(et, lens[b:b + 1]), 1, S, nh, hd, 1.0 / math.sqrt(hd))
    et.linear_dense(up(et, W["o"]), None, d1["z"], d1["out"], S, H, H)
    assert Hn.max_abs(d1["out"].numpy(), got[b * S:(b + 1) * S]) <= 1e-3


@pytest.mark.parametrize("B", [1, 4, 16])
def test_mha_block_config(et, B):
    """Attention core of the BERT-base block: S128, 12 heads x 64, right padding U{64..128}."""
    lens = torch.randint(64, 129, (B,), generator=Hn.rng(100 + B)).numpy()
    got, want = run_mha(et, B, 128, 12, 64, seed=50, lens=lens, single_buffer=True)
    err = Hn.max_abs(got, want)
    print(f"mha B={B} lens={lens.tolist()} max-abs={err:.2e}")
    assert err <= 2e-3


@pytest.mark.parametrize("B,S,nh,hd,causal", [(1, 128, 12, 64, True), (2, 512, 16, 64, False),
                                              (1, 384, 12, 64, False), (3, 32, 4, 32, False),
                                              (2, 48, 2, 128, True), (1, 16, 1, 64, False),
                                              (2, 272, 4, 64, True),
                                              # many workgroups per (sequence, head), several key blocks each
                                              (8, 512, 8, 64, False), (8, 512, 8, 64, True), (16, 256, 8, 32, True)])
def test_mha_shapes(et, B, S, nh, hd, causal):
    got, want = run_mha(et, B, S, nh, hd, seed=60, causal=causal)
    assert Hn.max_abs(got, want) <= 2e-3


@pytest.mark.parametrize("B,S,nh,hd,causal", [(2, 128, 4, 48, False), (1, 64, 3, 16, True), (2, 160, 2, 96, False),
                                              (1, 128, 5, 80, True), (1, 32, 2, 112, False),
                                              (2, 128, 4, 200, False),  # the reference example's heads (example/main.cu:24-31)
                                              (1, 160, 3, 256, True), (2, 48, 2, 136, False), (1, 64, 5, 40, True),
                                              (2, 128, 3, 72, False), (1, 272, 2, 168, False)])
def test_mha_head_sizes_between_template_sizes(et, B, S, nh, hd, causal):
    """Head sizes that are multiples of 8 but not 32/64/128/256 (the reference's kernels ask for hd % 16 == 0,
    Fused_attention/test/testfused.cu:22; its example has 200-wide heads), with right padding."""
    lens = [S - 7 * (b + 1) for b in range(B)]
    got, want = run_mha(et, B, S, nh, hd, seed=70, lens=lens, causal=causal)
    assert Hn.max_abs(got, want) <= 2e-3
    got, want = run_mha(et, B, S, nh, hd, seed=71, single_buffer=True)
    assert Hn.max_abs(got, want) <= 2e-3


def _random_mha_cases(n, seed):
    rng = np.random.default_rng(seed)
    cases = []
    for _ in range(n):
        S = 16 * int(rng.integers(1, 41))
        B, nh, hd = int(rng.integers(1, 7)), int(rng.integers(1, 9)), 16 * int(rng.integers(1, 9))
        kind = int(rng.integers(0, 4))  # 0 plain, 1 right padding, 2 causal, 3 additive mask with padding
        cases.append((B, S, nh, hd, kind, int(rng.integers(1, 1 << 30))))
    return cases


@pytest.mark.parametrize("B,S,nh,hd,kind,seed", _random_mha_cases(24, 20211116))
def test_mha_random_shapes(et, B, S, nh, hd, kind, seed):
    """Seeded random shapes: every head size from 16 to 128, 1 to 40 query tiles, plain, padded, causal and
    additively masked, separate and interleaved Q/K/V buffers."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, S + 1, B).astype(np.int32) if kind in (1, 3) else None
    # the mask is binary16 data: the oracle gets the same rounded values the kernel reads
    mask = (rng.standard_normal((S, S)) * 2.0).astype(np.float16).astype(np.float32) if kind == 3 else None
    got, want = run_mha(et, B, S, nh, hd, seed=seed & 0xFFFF, lens=lens, causal=kind == 2, mask=mask,
                        single_buffer=bool(seed & 1))
    if lens is not None:  # rows past a sequence's length are padding: not compared
        for b in range(B):
            got[b * S + lens[b]:(b + 1) * S] = 0
            want[b * S + lens[b]:(b + 1) * S] = 0
    assert Hn.max_abs(got, want) <= 2e-3


def test_mha_many_strips_with_padding(et):
    """Right padding at S = 256: lengths that end inside a key block, on a block boundary, inside a
    query strip, and a zero-length sequence (full blocks take the branch-free path, the last
    block of a padded sequence the masked one)."""
    B, S, nh, hd = 16, 256, 16, 64
    lens = [256, 1, 0, 129, 128, 200, 255, 17] * 2
    got, want = run_mha(et, B, S, nh, hd, seed=61, lens=lens)
    assert Hn.max_abs(got, want) <= 2e-3


@pytest.mark.parametrize("causal,padded", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("pad", [0, 4])
def test_mha_large_grid(et, causal, padded, pad):
    """Enough (sequence, head) pairs and queries that workgroups of 8 waves with two query tiles per
    wave (256 queries) are used where the 32 x 32 kernel is not (pad 4: rows of the result off 16 bytes); branch-free and masked key blocks, partial last
    blocks."""
    B, S, nh, hd = 32, 256, 16, 64
    lens = ([256, 3, 0, 129, 128, 250, 255, 17] * 4) if padded else None
    got, want = run_mha(et, B, S, nh, hd, seed=63, lens=lens, causal=causal, pad=pad)
    assert Hn.max_abs(got, want) <= 2e-3


# two rows: waves in turn; two tiles would be 128-wide heads' fourth and sixth, which have a form of one tile instead
LARGE_GRIDS = [(6, 768, 32, 64, False), (6, 768, 32, 64, True), (16, 128, 16, 128, False), (4, 384, 24, 128, True), (32, 256, 16, 128, False), (16, 512, 16, 128, True)]


@pytest.mark.parametrize("B,S,nh,hd,causal", LARGE_GRIDS)
@pytest.mark.parametrize("pad", [0, 4])
def test_mha_large_grid_shapes(et, B, S, nh, hd, causal, pad):
    lens = [S - (37 * b) % (S // 2) for b in range(B)]
    got, want = run_mha(et, B, S, nh, hd, seed=64, lens=lens, causal=causal, pad=pad)
    assert Hn.max_abs(got, want) <= 2e-3


# Forms that an additive mask keeps from the 32 x 32 kernel: eight waves with two tiles, eight with one, two, one
MASKED = [(32, 256, 16, 64, False), (6, 768, 32, 64, True), (32, 256, 16, 80, False), (16, 128, 16, 64, False), (16, 112, 16, 96, False), (16, 128, 16, 128, False),
          (64, 32, 8, 64, False), (64, 32, 8, 128, True), (150, 16, 12, 32, False)]


@pytest.mark.parametrize("B,S,nh,hd,causal", MASKED)
def test_mha_additive_mask_in_every_form(et, B, S, nh, hd, causal):
    mask = Hn.randn((S, S), 70, 1.0, np.float32)
    mask[torch.rand(S, S, generator=Hn.rng(71)).numpy() < 0.3] = -np.inf
    mask[:, 0] = 0.0  # every query keeps a key
    got, want = run_mha(et, B, S, nh, hd, seed=66, causal=causal, mask=mask.astype(np.float16).astype(np.float32), pad=4)
    assert Hn.max_abs(got, want) <= 2e-3


def test_mha_additive_mask_and_lens(et):
    B, S, nh, hd = 2, 128, 4, 64
    mask = Hn.randn((S, S), 70, 1.0, np.float32)
    mask[torch.rand(S, S, generator=Hn.rng(71)).numpy() < 0.3] = -np.inf
    mask[np.arange(S), np.arange(S)] = 0.0  # every query keeps at least itself ...
    mask[:, 0] = 0.0                        # ... and key 0, which survives any padding
    lens = np.array([128, 77])
    got, want = run_mha(et, B, S, nh, hd, seed=72, lens=lens, mask=mask)
    assert Hn.max_abs(got, want) <= 2e-3


def test_mha_padding_properties(et):
    """Padded keys get exactly zero weight: changing K/V rows beyond lens changes nothing,
    and each sequence of a batch equals the same sequence run alone."""
    B, S, nh, hd = 3, 128, 12, 64
    H = nh * hd
    lens = np.array([64, 100, 128], np.int32)
    q, k, v = Hn.randn((B * S, H), 80), Hn.randn((B * S, H), 81), Hn.randn((B * S, H), 82)
    k2, v2 = k.copy(), v.copy()
    for b in range(B):
        k2[b * S + lens[b]:(b + 1) * S] = np.float16(50.0)
        v2[b * S + lens[b]:(b + 1) * S] = np.float16(-1000.0)

    def run(qq, kk, vv, BB, ll):
        d_z = et.DeviceBuffer.empty((BB * S, H), np.float16)
        et.mha_fused(up(et, qq), up(et, kk), up(et, vv), H, H, H, d_z, H, None, up(et, ll), BB, S, nh, hd,
                     0.125)
        return d_z.numpy()

    base = run(q, k, v, B, lens)
    assert np.array_equal(base, run(q, k2, v2, B, lens))
    for b in range(B):
        sl = slice(b * S, (b + 1) * S)
        alone = run(q[sl], k[sl], v[sl], 1, lens[b:b + 1])
        assert np.array_equal(base[sl], alone)
    assert np.all(np.isfinite(base.astype(np.float32)))


@pytest.mark.parametrize("B,S,nh,hd,causal", [(16, 128, 12, 64, False), (16, 512, 8, 64, True), (12, 400, 8, 128, False), (40, 272, 4, 200, False)])
def test_mha_sequences_of_a_large_batch(et, B, S, nh, hd, causal):
    """A sequence of a large batch against the same sequence alone, whose keys the launch sums in other parts: the probabilities enter the product rounded to
    binary16 against other maxima (2^-11 of each on either side) and so do the results, 2^-9 of max |V| < 5.5, 1e-3 of the norm.  Batches that sum
    in the same parts agree bit for bit."""
    H = nh * hd
    q, k, v = (Hn.randn((2 * B * S, H), 80 + i) for i in range(3))
    lens = np.array([S - (29 * b) % S for b in range(2 * B)], np.int32)

    def run(first, n):
        rows = slice(first * S, (first + n) * S)
        d_z = up(et, np.full((n * S, H), np.nan, np.float16))
        et.mha_fused(up(et, q[rows]), up(et, k[rows]), up(et, v[rows]), H, H, H, d_z, H, None, up(et, lens[first:first + n]), n, S, nh, hd, hd ** -0.5,
                     et.MHA_CAUSAL if causal else 0)
        return d_z.numpy()

    both, half = run(0, 2 * B), run(0, B)
    assert np.array_equal(both[:B * S], half)
    for b in (0, 1, B - 1):
        alone = run(b, 1).astype(np.float32)
        batch = half[b * S:(b + 1) * S].astype(np.float32)
        assert np.abs(alone - batch).max() <= 1.1e-2 and np.linalg.norm(alone - batch) <= 1e-3 * np.linalg.norm(alone)


def test_mha_zero_length_sequence_gives_zeros(et):
    B, S, nh, hd = 2, 32, 2, 64
    got, _ = run_mha(et, B, S, nh, hd, seed=90, lens=np.array([0, 32]))
    assert np.all(got[:S] == 0)


def test_mha_rejects_bad_args(et):
    d = et.DeviceBuffer.empty((128, 768), np.float16)
    f = et.lib().et_mha_fused_f16
    args = lambda S, hd, ld: (d.ptr, d.ptr, d.ptr, ld, ld, ld, d.ptr, ld, None, None, 1, S, 12, hd, 0.125, 0, None)
    assert f(*args(120, 64, 768)) == et.ET_ERR_UNSUPPORTED   # S % 16
    assert f(*args(128, 44, 768)) == et.ET_ERR_UNSUPPORTED   # head dim not a multiple of 8
    assert f(*args(128, 264, 4096)) == et.ET_ERR_UNSUPPORTED  # head dim above 256
    assert f(*args(128, 64, 512)) == et.ET_ERR_INVALID_ARG   # stride < nh*hd
    assert f(None, d.ptr, d.ptr, 768, 768, 768, d.ptr, 768, None, None, 1, 128, 12, 64, 0.125, 0, None) == et.ET_ERR_INVALID_ARG


# ---------------------------------------------------------------- layer ------

@pytest.mark.parametrize("B,lens", [(1, None), (2, [100, 128])])
def test_encoder_layer_via_kernels(et, B, lens):
    err = Hn.run_layer_case(et, H=768, nh=12, dimFF=3072, S=128, B=B, sparsity=0.8, seed=3, lens=lens)
    print(f"layer B={B} max-abs={err:.2e}")
    assert err <= TOL_F16
