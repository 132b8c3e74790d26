"""What the performance of this engine is measured on: the work its users give it, through the public entry
points of the package (``scpaper-2021_amd/__init__.py``) and of the C ABI behind it (``include/et_abi.h``).

Encoder stacks come first, since a forward of a pruned stack is what the engine is for: from one sequence of
128 tokens (latency and launches) over the batch the headline benchmark runs to thousands of token rows, tile-sparse
and dense, both residual precisions, ragged row counts, and the binary32 twin.  The single calls after them are what
a program uses that assembles its own layers: fused attention, a tile-sparse, a dense and a row- or column-pruned
Linear, and SkipLayerNorm.  The engine is inference only, so every case is a forward.

Every call goes to one stream of the program's own, as a server's would; inputs, weights, plans and outputs stay on
the device between calls.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__ as entry

et = entry.load_package()

_stream = None


def stream():
    """The program's stream, created with the first state."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


# ---------------------------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------------------------

def encoder(H, nh, FF, layers, B, S, sparsity, mixed, **options):
    """A stack of encoder layers on B sequences of S tokens; sparsity 0: dense weights (mixed: the residual stream is
    binary32 inside the stack, else every activation is binary16)."""
    case = {"kind": "encoder", "H": H, "nh": nh, "FF": FF, "layers": layers, "B": B, "S": S, "sparsity": sparsity, "mixed": mixed,
            "aware": False, "padded": False, "causal": False, "act": "gelu"}
    case.update(options)
    return case


def listed():
    return [
        # One request at a time: BERT-base, one sequence, nothing to batch it with (the sweep of the class layer's
        # Table 2 program).  Launches and latency.
        dict(encoder(768, 12, 3072, 12, 1, 128, 0.8, 1), name="base-1x128-tile80"),
        # The headline workload of bench.py: eight sequences, attention-aware pruning of a quarter of V and O.
        dict(encoder(768, 12, 3072, 12, 8, 128, 0.8, 1, aware=True), name="base-8x128-tile80-aware"),
        # A full batch of requests of unequal length: throughput.
        dict(encoder(768, 12, 3072, 12, 64, 128, 0.8, 1, padded=True), name="base-64x128-tile80-padded"),
        # Long documents through BERT-large at 90 %, padded.
        dict(encoder(1024, 16, 4096, 24, 4, 512, 0.9, 1, padded=True), name="large-4x512-tile90-padded"),
        # The six-layer model at light pruning, a ragged batch (528 token rows), activations as the reference stores
        # them.
        dict(encoder(768, 12, 3072, 6, 3, 176, 0.6, 0, act="relu"), name="distil-3x176-tile60"),
        # The unpruned model a pruned one is compared with.
        dict(encoder(768, 12, 3072, 12, 16, 128, 0.0, 0), name="base-16x128-dense"),
        # The binary32 twin: checking a pruned model's values without binary16 rounding.
        {"kind": "encoder_f32", "H": 768, "nh": 12, "FF": 3072, "layers": 6, "B": 2, "S": 128, "sparsity": 0.8, "padded": True,
         "name": "f32-base-2x128-tile80"},
        # Long-context attention on its own.
        {"kind": "attention", "B": 16, "S": 2048, "nh": 16, "hd": 64, "padded": False, "causal": False, "name": "attention-16x2048"},
        # The tile-sparse FFN down-projection of a mid-sized batch, in the container's own layout.
        {"kind": "tile", "T": 4096, "in": 3072, "out": 768, "sparsity": 0.8, "act": "none", "name": "tile-4096-3072-768"},
        # A dense projection large enough that only the matrix cores count.
        {"kind": "dense", "T": 8192, "in": 4096, "out": 4096, "act": "none", "name": "dense-8192-4096-4096"},
        # The FFN up-projection with half of its input features pruned.
        {"kind": "pruned", "side": "col", "T": 2048, "in": 768, "out": 3072, "sparsity": 0.5, "act": "gelu", "name": "colpruned-2048-768-3072"},
        # SkipLayerNorm over a large batch: memory.
        {"kind": "norm", "rows": 65536, "H": 768, "skip": True, "name": "skipln-65536x768"},
    ]


def _log(rng, lo, hi, step):
    """A multiple of step between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["encoder"] * 5 + ["attention", "attention", "tile", "dense", "pruned", "norm", "encoder_f32"])
    act = rng.choice(["none", "relu", "gelu"])
    if kind == "encoder":
        H, nh, FF = rng.choice([(768, 12, 3072), (768, 12, 3072), (1024, 16, 4096), (512, 8, 2048), (384, 6, 1536), (800, 4, 208)])
        S = _log(rng, 16, 512, 16)
        B = _log(rng, 1, max(1, min(64, 8192 // S)), 1)
        # at most the token rows x layers x weights of the listed stacks
        layers = rng.randint(2, max(2, min(12, int(12 * 8192 * 768 * 768 / (B * S * H * H)))))
        sparsity = rng.choice([0.0, 0.4, 0.6, 0.7, 0.8, 0.8, 0.9, 0.95])
        if sparsity < 0.6:
            layers = min(layers, max(2, 20480 * 768 * 768 // (B * S * H * H)))
        return encoder(H, nh, FF, layers, B, S, sparsity, rng.choice([0, 1, 1]), padded=rng.random() < 0.5, causal=rng.random() < 0.25,
                       act=rng.choice(["relu", "gelu"]))
    if kind == "encoder_f32":
        S = _log(rng, 16, 256, 16)
        return {"kind": kind, "H": 768, "nh": 12, "FF": 3072, "layers": rng.randint(1, 6), "B": _log(rng, 1, max(1, 512 // S), 1), "S": S,
                "sparsity": rng.choice([0.0, 0.5, 0.8, 0.9]), "padded": rng.random() < 0.5}
    if kind == "attention":
        S = _log(rng, 16, 2048, 16)
        nh, hd = rng.choice([(12, 64), (16, 64), (8, 128), (4, 200), (12, 32), (10, 80)])
        return {"kind": kind, "B": _log(rng, 1, max(1, min(64, 32768 // S)), 1), "S": S, "nh": nh, "hd": hd, "padded": rng.random() < 0.4,
                "causal": rng.random() < 0.4}
    if kind == "tile":
        n_in, n_out = rng.choice([(768, 768), (768, 3072), (3072, 768), (1024, 4096), (4096, 1024), (1024, 1024), (768, 2304), (208, 800)])
        return {"kind": kind, "T": _log(rng, 16, 16384, 16), "in": n_in, "out": n_out, "sparsity": rng.choice([0.5, 0.7, 0.8, 0.9, 0.95]), "act": act}
    if kind == "dense":
        return {"kind": kind, "T": _log(rng, 16, 8192, 16), "in": _log(rng, 208, 4096, 16), "out": _log(rng, 208, 4096, 16), "act": act}
    if kind == "pruned":
        n_in, n_out = rng.choice([(768, 768), (768, 3072), (3072, 768), (1024, 4096), (2048, 2048)])
        return {"kind": kind, "side": rng.choice(["row", "col"]), "T": _log(rng, 16, 8192, 16), "in": n_in, "out": n_out,
                "sparsity": rng.choice([0.3, 0.5, 0.7, 0.9]), "act": act}
    return {"kind": "norm", "rows": _log(rng, 16, 65536, 1), "H": rng.choice([256, 384, 768, 768, 800, 1024]), "skip": rng.random() < 0.7}


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------

ACT = {"none": et.ACT_NONE, "relu": et.ACT_RELU, "gelu": et.ACT_GELU}


class Rng:
    """Seeded values made on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.seed = seed * 1000003

    def next_seed(self):
        self.seed += 1
        return self.seed

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(dtype)

    def lens(self, B, S):
        """Sequence lengths from half of S to S, one of them full."""
        n = torch.randint(S // 2, S + 1, (B,), generator=self.g, device="cuda").to(torch.int32)
        n[-1] = S
        return n


def kept_tiles(n_in, n_out, sparsity):
    return et.lib().et_fmt_kept_count((n_out // 16) * (n_in // 16), sparsity)


def tile_pattern(r, n_in, n_out, sparsity, dead_rows=(), dead_cols=()):
    """Row pointers and column indices of a seeded random tile pattern; no tile in the dead block-rows and -columns."""
    nc = n_in // 16
    total = (n_out // 16) * nc
    perm = np.zeros(total, np.int64)
    et.check(et.lib().et_fmt_permutation(total, r.next_seed(), perm.ctypes.data))
    if len(dead_rows) or len(dead_cols):
        perm = perm[~np.isin(perm // nc, dead_rows) & ~np.isin(perm % nc, dead_cols)]
    kept = perm[:kept_tiles(n_in, n_out, sparsity)]
    kept = kept[np.argsort(kept // nc, kind="stable")]
    row_ptr = np.concatenate([[0], np.cumsum(np.bincount(kept // nc, minlength=n_out // 16))])
    return row_ptr.astype(np.int32), (kept % nc).astype(np.int32)


def layer_matrices(H, FF):
    return ((et.W_QKV, H, 3 * H), (et.W_O, H, H), (et.W_FF1, H, FF), (et.W_FF2, FF, H))


def prepare_encoder(c, r):
    H, nh, FF, B, S = c["H"], c["nh"], c["FF"], c["B"], c["S"]
    model = et.Model(H, nh, FF, S, c["layers"], batch=B, act=ACT[c["act"]], causal=c["causal"], use_graph=True, mixed=c["mixed"])
    per_head = H // nh // 16
    dead = [h * per_head + per_head - 1 - i for h in range(nh) for i in range(per_head // 4)] if c["aware"] else []
    for layer in range(c["layers"]):
        for which, n_in, n_out in layer_matrices(H, FF):
            bias = r.normal(n_out, std=0.02)
            if c["sparsity"] == 0.0:
                model.set_dense(layer, which, r.normal(n_out, n_in, std=0.02).cpu().numpy(), bias.cpu().numpy())
                continue
            rows = [2 * (H // 16) + b for b in dead] if which == et.W_QKV else []
            if rows:
                bias.view(-1, 16)[rows] = 0
            row_ptr, col = tile_pattern(r, n_in, n_out, c["sparsity"], rows, dead if which == et.W_O else [])
            model.set_bsr16(layer, which, row_ptr, col, r.normal(len(col), 256, std=0.02).cpu().numpy(), bias.cpu().numpy())
        for k in (0, 1):
            model.set_norm(layer, k, r.normal(H, std=0.1, mean=1.0).cpu().numpy(), r.normal(H, std=0.1).cpu().numpy())
    if c["padded"]:
        model.set_lens(r.lens(B, S).cpu().numpy())
    model.finalize()
    x = r.normal(B * S, H)
    return {"model": model, "x": x, "out": torch.empty_like(x)}


class ModelF32:
    """Owner of an et_model_f32 handle."""

    def __init__(self, desc):
        h = ctypes.c_void_p()
        et.check(et.lib().et_model_f32_create(ctypes.byref(desc), ctypes.byref(h)))
        self.handle = h.value

    def __del__(self):
        et.lib().et_model_f32_destroy(self.handle)


def prepare_encoder_f32(c, r):
    H, nh, FF, B, S = c["H"], c["nh"], c["FF"], c["B"], c["S"]
    lib = et.lib()
    model = ModelF32(et.ModelDesc(H, H, S, nh, FF, H, c["layers"], B, et.ACT_GELU, 1e-5, 0, 1, 0))

    def host(*shape, std=1.0, mean=0.0):
        return r.normal(*shape, std=std, mean=mean, dtype=torch.float32).cpu().numpy()

    for layer in range(c["layers"]):
        for which, n_in, n_out in layer_matrices(H, FF):
            bias = host(n_out, std=0.02)
            if c["sparsity"] == 0.0:
                w = host(n_out, n_in, std=0.02)
                et.check(lib.et_model_f32_set_dense(model.handle, layer, which, w.ctypes.data, bias.ctypes.data))
            else:
                row_ptr, col = tile_pattern(r, n_in, n_out, c["sparsity"])
                w = host(len(col), 256, std=0.02)
                et.check(lib.et_model_f32_set_bsr16(model.handle, layer, which, row_ptr.ctypes.data, col.ctypes.data, w.ctypes.data, len(col),
                                                    bias.ctypes.data))
        for k in (0, 1):
            g, b = host(H, std=0.1, mean=1.0), host(H, std=0.1)
            et.check(lib.et_model_f32_set_norm(model.handle, layer, k, g.ctypes.data, b.ctypes.data))
    if c["padded"]:
        lens = r.lens(B, S).cpu().numpy()
        et.check(lib.et_model_f32_set_lens(model.handle, lens.ctypes.data))
    et.check(lib.et_model_f32_finalize(model.handle))
    x = r.normal(B * S, H, dtype=torch.float32)
    return {"model": model, "x": x, "out": torch.empty_like(x)}


def prepare(case, seed):
    c, r = case, Rng(seed)
    kind = c["kind"]
    if kind == "encoder":
        state = prepare_encoder(c, r)
    elif kind == "encoder_f32":
        state = prepare_encoder_f32(c, r)
    elif kind == "attention":  # Q, K and V as the slices of one projection's result
        T, H = c["B"] * c["S"], c["nh"] * c["hd"]
        state = {"qkv": r.normal(T, 3 * H), "out": torch.empty(T, H, dtype=torch.float16, device="cuda"),
                 "lens": r.lens(c["B"], c["S"]) if c["padded"] else None}
    elif kind == "norm":
        rows, H = c["rows"], c["H"]
        state = {"x": r.normal(rows, H), "skip": r.normal(rows, H) if c["skip"] else None, "gamma": r.normal(H, std=0.1, mean=1.0),
                 "beta": r.normal(H, std=0.1), "out": torch.empty(rows, H, dtype=torch.float16, device="cuda")}
    else:  # the Linear layers
        T, n_in, n_out = c["T"], c["in"], c["out"]
        state = {"x": r.normal(T, n_in), "bias": r.normal(n_out, std=0.02), "out": torch.empty(T, n_out, dtype=torch.float16, device="cuda")}
        if kind == "tile":
            row_ptr, col = tile_pattern(r, n_in, n_out, c["sparsity"])
            state.update(row_ptr=torch.from_numpy(row_ptr).cuda(), col=torch.from_numpy(col).cuda(), w=r.normal(len(col), 256, std=0.02))
        elif kind == "dense":
            state.update(w=r.normal(n_out, n_in, std=0.02))
        else:
            ids, n = np.zeros(max(n_in, n_out), np.int32), ctypes.c_int()
            gen, width = (et.lib().et_fmt_row_ids, n_out) if c["side"] == "row" else (et.lib().et_fmt_col_ids, n_in)
            et.check(gen(width, c["sparsity"], r.next_seed(), ids.ctypes.data, ctypes.byref(n)))
            n = n.value // 16 * 16
            ids = torch.from_numpy(ids[:n].copy()).cuda()
            if c["side"] == "row":
                state.update(ids=ids, n=n, w=r.normal(n, n_in, std=0.02))
            else:
                state.update(ids=ids, n=n, w=r.normal(n_out, n, std=0.02), gathered=torch.empty(T, n, dtype=torch.float16, device="cuda"))
    state["case"], state["stream"] = c, stream()
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------------------------

def run(state):
    s, c, out, on = state, state["case"], state["out"], state["stream"]
    kind = c["kind"]
    if kind == "encoder":
        s["model"].forward(out.data_ptr(), s["x"].data_ptr(), on)
    elif kind == "encoder_f32":
        et.check(et.lib().et_model_f32_forward(s["model"].handle, out.data_ptr(), s["x"].data_ptr(), on))
    elif kind == "attention":
        H, q = c["nh"] * c["hd"], s["qkv"].data_ptr()
        et.mha_fused(q, q + 2 * H, q + 4 * H, 3 * H, 3 * H, 3 * H, out.data_ptr(), H, None,
                     None if s["lens"] is None else s["lens"].data_ptr(), c["B"], c["S"], c["nh"], c["hd"], c["hd"] ** -0.5,
                     et.MHA_CAUSAL if c["causal"] else 0, on)
    elif kind == "norm":
        if s["skip"] is not None:
            et.skip_layernorm(out.data_ptr(), s["x"].data_ptr(), s["skip"].data_ptr(), s["gamma"].data_ptr(), s["beta"].data_ptr(), c["rows"],
                              c["H"], 1e-5, on)
        else:
            et.layernorm(out.data_ptr(), s["x"].data_ptr(), s["gamma"].data_ptr(), s["beta"].data_ptr(), c["rows"], c["H"], 1e-5, on)
    elif kind == "tile":
        et.linear_bsr16(s["row_ptr"].data_ptr(), s["col"].data_ptr(), s["w"].data_ptr(), s["bias"].data_ptr(), s["x"].data_ptr(),
                        out.data_ptr(), c["T"], c["in"], c["out"], ACT[c["act"]], on)
    elif kind == "dense":
        et.linear_dense(s["w"].data_ptr(), s["bias"].data_ptr(), s["x"].data_ptr(), out.data_ptr(), c["T"], c["in"], c["out"], ACT[c["act"]], on)
    elif c["side"] == "row":
        et.check(et.lib().et_linear_rowpruned_f16(s["w"].data_ptr(), s["ids"].data_ptr(), s["n"], s["bias"].data_ptr(), s["x"].data_ptr(),
                                                  out.data_ptr(), c["T"], c["in"], c["out"], ACT[c["act"]], on))
    else:
        et.check(et.lib().et_linear_colpruned_ws_f16(s["w"].data_ptr(), s["ids"].data_ptr(), s["n"], s["bias"].data_ptr(), s["x"].data_ptr(),
                                                     out.data_ptr(), s["gathered"].data_ptr(), c["T"], c["in"], c["out"], ACT[c["act"]], on))
    return out


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, and how near another correct implementation comes
# ---------------------------------------------------------------------------------------------------------------

def attention_flops(c):
    """Scores and weighted sum of B sequences; padded keys (a quarter on average) and keys above the diagonal are not needed."""
    pairs = c["S"] * c["S"] * (0.5 if c.get("causal") else 1.0) * (0.75 if c.get("padded") else 1.0)
    return 4.0 * c["B"] * pairs * (c["H"] if "H" in c else c["nh"] * c["hd"])


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("encoder", "encoder_f32"):
        size = 4 if kind == "encoder_f32" else 2
        T, weights, flops = c["B"] * c["S"], 0, attention_flops(c)
        for _, n_in, n_out in layer_matrices(c["H"], c["FF"]):
            values = n_in * n_out if c["sparsity"] == 0.0 else 256 * kept_tiles(n_in, n_out, c["sparsity"])
            weights += size * (values + n_out)
            flops += 2.0 * values * T
        return {"bytes": c["layers"] * (weights + 4 * size * c["H"]) + 2 * size * T * c["H"], "flops": c["layers"] * flops}
    if kind == "attention":
        return {"bytes": 8 * c["B"] * c["S"] * c["nh"] * c["hd"], "flops": attention_flops(c)}
    if kind == "norm":
        return {"bytes": (6 if c["skip"] else 4) * c["rows"] * c["H"] + 4 * c["H"], "flops": 0}
    T, n_in, n_out = c["T"], c["in"], c["out"]
    x, y = T * n_in, T * n_out
    if kind == "tile":
        values = 256 * kept_tiles(n_in, n_out, c["sparsity"])
    elif kind == "dense":
        values = n_in * n_out
    else:
        kept = int((n_out if c["side"] == "row" else n_in) * (1 - c["sparsity"]))
        values = kept * (n_in if c["side"] == "row" else n_out)
        x = x if c["side"] == "row" else T * kept
    return {"bytes": 2 * (x + y + values + n_out), "flops": 2.0 * values * T}


def tolerance(case):
    """binary16 results carry 2^-11 of rounding each (3e-4 in the mean); a stack rounds its operands, and its residual
    where that is binary16, once per sublayer.  binary32 sums agree to 1e-5."""
    if case["kind"] == "encoder":
        return {"rel": 5e-3}
    if case["kind"] == "encoder_f32":
        return {"rel": 1e-5}
    return {"rel": 2e-3 if case["kind"] == "attention" else 1e-3}
