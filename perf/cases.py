"""The work a program built on this library has it do, as cases that can be timed and compared.

Every case goes through the public entry points: Engine, Exl3Linear.run_bufs, ne_exl3_lin_run_multi, hc_read,
MoeLayer.run_bufs and MoeLayer.run_hc, on device buffers, one call after another on the library's stream, as a decode
loop or a prefill loop calls them. Shapes are those of the repository's benchmark and tests: hidden 2048 x inter 512
with its trunk (q 4096, k and v 512, o; vocabulary 151936) and the reference's own hidden 2560 x inter 640 with its
trunk (10240, 640) and hyper-connection mixes (4 x 2560 -> 320 -> 4 x 2560); 512 experts, top-10.

A pass of a small case covers several layers, each with its own weights, so that weights come from HBM as they do in a
model and not from the last-level cache.
"""
import ctypes
import math

import numpy as np
import torch

NE, TOPK = 512, 10

# trunk shapes by hidden size: the linears of one launch (same input), then the linear back to the hidden size
TRUNK = {2048: ((4096, 512, 512), 4096), 2560: ((10240, 640, 640), 10240)}
MOE = {"2048x512": (2048, 512), "2560x640": (2560, 640), "1024x256": (1024, 256)}


def listed():
    return [
        # one token of a decode loop: the attention linears (q, k, v in one launch, then o) of eight layers
        {"name": "trunk_1row", "kind": "trunk", "hid": 2048, "K": 6, "rows": 1, "layers": 8},
        # the same for the drafts of several sequences verified together
        {"name": "trunk_16rows", "kind": "trunk", "hid": 2048, "K": 6, "rows": 16, "layers": 4},
        # the vocabulary head for one token, and for a ragged batch of drafts
        {"name": "head_1row", "kind": "head", "inp": 2048, "out": 151936, "K": 8, "rows": 1},
        {"name": "head_13rows", "kind": "head", "inp": 2048, "out": 151936, "K": 8, "rows": 13},
        # the hyper-connection read in front of the MoE block, one token, eight layers
        {"name": "hc_read_1row", "kind": "hc", "hid": 2560, "lr": 320, "K": 6, "rows": 1, "layers": 8},
        # the MoE layer of one token, eight layers: the benchmark's shape, and the reference's with its 8-bit shared
        # expert and the hyper-connection write
        {"name": "moe_1row", "kind": "moe", "shape": "2048x512", "K": 5, "shared": "exl3", "Ks": 5, "hc": False,
         "rows": 1, "layers": 8},
        {"name": "moe_1row_q8_hc", "kind": "moe", "shape": "2560x640", "K": 5, "shared": "q8", "Ks": 0, "hc": True,
         "rows": 1, "layers": 8},
        # speculative verify of one sequence's drafts, the MTP head's bit widths
        {"name": "moe_6rows_k4", "kind": "moe", "shape": "2048x512", "K": 4, "shared": "exl3", "Ks": 6, "hc": False,
         "rows": 6, "layers": 2},
        # a batch of sequences decoding together
        {"name": "moe_48rows", "kind": "moe", "shape": "2048x512", "K": 5, "shared": "exl3", "Ks": 5, "hc": False,
         "rows": 48, "layers": 1},
        # a short prompt, and the odd last chunk of a long one at the reference's shape
        {"name": "moe_300rows_q8_hc", "kind": "moe", "shape": "2560x640", "K": 5, "shared": "q8", "Ks": 0, "hc": True,
         "rows": 300, "layers": 1},
        {"name": "moe_1111rows", "kind": "moe", "shape": "2048x512", "K": 5, "shared": "exl3", "Ks": 5, "hc": False,
         "rows": 1111, "layers": 1},
        # a full prefill chunk
        {"name": "moe_4096rows", "kind": "moe", "shape": "2048x512", "K": 5, "shared": "exl3", "Ks": 5, "hc": False,
         "rows": 4096, "layers": 1},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["trunk", "head", "hc", "moe", "moe", "moe", "moe"])
    if kind == "trunk":
        rows = _log_int(rng, 1, 32)
        return {"kind": kind, "hid": rng.choice([2048, 2560]), "K": rng.choice([4, 5, 6, 8]), "rows": rows,
                "layers": rng.randint(3, 8)}
    if kind == "head":
        return {"kind": kind, "inp": rng.choice([2048, 2560]), "out": 16 * _log_int(rng, 2000, 9000),
                "K": rng.choice([5, 6, 8]), "rows": _log_int(rng, 1, 32)}
    if kind == "hc":
        return {"kind": kind, "hid": rng.choice([2048, 2560]), "lr": 320, "K": rng.choice([5, 6, 8]),
                "rows": _log_int(rng, 1, 32), "layers": rng.randint(3, 8)}
    shape = rng.choice(["2048x512", "2560x640", "1024x256"])
    # as many decode and verify calls as batches and prefill chunks
    rows = _log_int(rng, 1, 32) if rng.random() < 0.4 else _log_int(rng, 33, 2400 if shape == "2560x640" else 4000)
    shared = rng.choice(["exl3", "q8"])
    return {"kind": kind, "shape": shape, "K": rng.choice([4, 5, 5, 6]), "shared": shared,
            "Ks": rng.choice([4, 5, 6]) if shared == "exl3" else 0, "hc": rng.random() < 0.5, "rows": rows,
            "layers": rng.randint(4, 8) if rows == 1 else 2 if rows <= 8 else 1}


# ---------------------------------------------------------------------------------------------------- a program's side
_engine = None


def _eng():
    global _engine
    if _engine is None:
        import ijah_amd
        _engine = ijah_amd.load_engine()
    return _engine


class _Bytes:
    """A device buffer's memory, for torch."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 3, "strides": None,
                                         "data": (int(buf.gpu_address()), False)}


def _view(buf, shape, typestr="<f4"):
    return torch.as_tensor(_Bytes(buf, shape, typestr), device="cuda")


def _buf(t):
    """A device buffer of the library with the tensor's bytes."""
    b = _eng().alloc(t.numel() * t.element_size())
    kind = {torch.float32: "<f4", torch.int16: "<i2"}[t.dtype]
    _view(b, t.shape, kind).copy_(t)
    return b


def _out(*shape):
    b = _eng().alloc(4 * int(np.prod(shape)))
    v = _view(b, shape)
    v.zero_()
    return b, v


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _bf16_values(g, *shape):
    """activations as the model's blocks hand them on: f32 holding bf16 values"""
    return _normal(g, *shape).bfloat16().float()


def _scales(g, n):
    """a channel's scale and sign, fp16"""
    m = (1 + 0.1 * _normal(g, n)).abs()
    s = torch.randint(0, 2, (n,), generator=g, device="cuda") * 2 - 1
    return (m * s).half()


def _lin_arrays(g, inp, out, K):
    """trellis int16 [in/16][out/16][16 K], suh, svh, on the GPU (every bit pattern is a valid trellis); the output
    scales carry the weights' 1 / sqrt(in), so that outputs are of the inputs' size"""
    t = torch.randint(-32768, 32768, (inp // 16, out // 16, 16 * K), generator=g, device="cuda", dtype=torch.int16)
    return t, _scales(g, inp), (_scales(g, out).float() / math.sqrt(inp)).half()


def _lin(arrays):
    t, su, sv = arrays
    return _eng().exl3_linear(t.cpu().numpy().view(np.uint16), su.cpu().numpy(), sv.cpu().numpy())


def _trunk_arrays(case, g):
    outs, back = TRUNK[case["hid"]]
    return [([_lin_arrays(g, case["hid"], o, case["K"]) for o in outs], _lin_arrays(g, back, case["hid"], case["K"]),
             _bf16_values(g, case["rows"], case["hid"]), _bf16_values(g, case["rows"], back))
            for _ in range(case["layers"])]


def _hc_arrays(case, g):
    hid, lr, K, R = case["hid"], case["lr"], case["K"], case["rows"]
    return [{"down": _lin_arrays(g, 4 * hid, lr, K), "up": _lin_arrays(g, lr, 4 * hid, K),
             "h": _bf16_values(g, R, 4, hid), "norm": (1 + 0.1 * _normal(g, 4 * hid)).bfloat16(),
             "inject": (_normal(g, 4, 4 * hid) / 100).bfloat16()} for _ in range(case["layers"])]


def _moe_inputs(case, g):
    hid, _ = MOE[case["shape"]]
    got = []
    for _ in range(case["layers"]):
        d = {"x": _bf16_values(g, case["rows"], hid)}
        if case["hc"]:  # the four residual streams and the read's gates (2 sigmoid, so around 1)
            d["h"] = _bf16_values(g, case["rows"], 4, hid)
            d["inj"] = torch.cat([(1 + 0.1 * _normal(g, case["rows"], 4)).bfloat16().float(),
                                  torch.ones(case["rows"], 4, device="cuda")], 1).contiguous()
        got.append(d)
    return got


def _moe_seed(seed, layer):
    return (seed % 1000003) * 64 + layer


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "trunk":
        state = []
        for qkv, o, x, a in _trunk_arrays(case, g):
            lins, n = [_lin(w) for w in qkv], len(qkv)
            xb, ab = _buf(x), _buf(a)
            ys = [_out(case["rows"], m.out) for m in lins]
            back = _lin(o)
            yb, yv = _out(case["rows"], back.out)
            state.append({"lins": lins, "n": n, "x": xb, "a": ab, "ys": ys, "back": back, "y": yb,
                          "ptr": (ctypes.c_void_p * n)(*[m.ptr for m in lins]),
                          "xp": (ctypes.c_void_p * n)(*[xb.ptr] * n), "yp": (ctypes.c_void_p * n)(*[b.ptr for b, _ in ys]),
                          "zero": (ctypes.c_uint64 * n)(), "views": [v for _, v in ys] + [yv]})
    elif kind == "head":
        w = _lin_arrays(g, case["inp"], case["out"], case["K"])
        yb, yv = _out(case["rows"], case["out"])
        state = [{"lin": _lin(w), "x": _buf(_bf16_values(g, case["rows"], case["inp"])), "y": yb, "views": [yv]}]
    elif kind == "hc":
        state = []
        for d in _hc_arrays(case, g):
            mix, mv = _out(case["rows"], case["lr"])
            inj, iv = _out(case["rows"], 8)
            out, ov = _out(case["rows"], case["hid"])
            state.append({"down": _lin(d["down"]), "up": _lin(d["up"]), "h": _buf(d["h"]),
                          "norm": _buf(d["norm"].view(torch.int16)), "inject": _buf(d["inject"].view(torch.int16)),
                          "mix": mix, "inj": inj, "out": out, "views": [mv, iv, ov]})
    else:
        hid, inter = MOE[case["shape"]]
        state = []
        for i, d in enumerate(_moe_inputs(case, g)):
            m = _eng().moe_synth(hid, inter, NE, TOPK, case["K"], "q8" if case["shared"] == "q8" else True,
                                 case["Ks"] or None, seed=_moe_seed(seed, i))
            yb, yv = _out(case["rows"], hid)
            s = {"moe": m, "x": _buf(d["x"]), "y": yb, "views": [yv]}
            if case["hc"]:
                s["h"], s["inj"] = _buf(d["h"]), _buf(d["inj"])
                s["hout"], hv = _out(case["rows"], 4, hid)
                s["views"].append(hv)
            state.append(s)
    torch.cuda.synchronize()
    return {"kind": kind, "rows": case["rows"], "hc": case.get("hc", False), "layers": state,
            "views": [s["views"] for s in state]}


def run(state):
    R, kind = state["rows"], state["kind"]
    if kind == "trunk":
        eng = _eng()
        for s in state["layers"]:
            if eng.lib.ne_exl3_lin_run_multi(s["ptr"], s["n"], R, s["xp"], s["zero"], s["yp"], s["zero"], None):
                raise RuntimeError(eng.last_error())
            s["back"].run_bufs(R, s["a"], s["y"])
    elif kind == "head":
        s = state["layers"][0]
        s["lin"].run_bufs(R, s["x"], s["y"])
    elif kind == "hc":
        from ijah_amd.engine import hc_read
        for s in state["layers"]:
            hc_read(s["down"], s["up"], R, s["h"], s["norm"], s["inject"], s["mix"], s["inj"], s["out"])
    elif state["hc"]:
        for s in state["layers"]:
            s["moe"].run_hc(R, s["x"], s["y"], s["h"], s["inj"], s["hout"])
    else:
        for s in state["layers"]:
            s["moe"].run_bufs(R, s["x"], s["y"])
    return state["views"]


# ---------------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    """weights, inputs and outputs each once; two operations per weight and row"""
    R, L = case["rows"], case.get("layers", 1)

    def lin(i, o, K):
        return i * o * K / 8 + 2 * (i + o)

    if case["kind"] == "trunk":
        hid, (outs, back) = case["hid"], TRUNK[case["hid"]]
        b = sum(lin(hid, o, case["K"]) for o in outs) + lin(back, hid, case["K"])
        n = hid * sum(outs) + back * hid
        b += 4 * R * (hid + sum(outs) + back + hid)
    elif case["kind"] == "head":
        n = case["inp"] * case["out"]
        b = lin(case["inp"], case["out"], case["K"]) + 4 * R * (case["inp"] + case["out"])
    elif case["kind"] == "hc":
        hid, lr = case["hid"], case["lr"]
        n = 8 * hid * lr
        b = lin(4 * hid, lr, case["K"]) + lin(lr, 4 * hid, case["K"]) + 2 * 20 * hid + 4 * R * (4 * hid + lr + 8 + hid)
    else:
        hid, inter = MOE[case["shape"]]
        w = 3 * hid * inter
        touched = NE * (1 - (1 - TOPK / NE) ** R)  # experts that R rows of independent tokens meet
        b = touched * (w * case["K"] / 8 + 6 * (hid + inter)) + 2 * NE * hid
        b += w * 33 / 32 if case["shared"] == "q8" else w * case["Ks"] / 8 + 6 * (hid + inter)
        b += 4 * R * hid * (10 if case["hc"] else 2)
        n = w * (TOPK + 1) + NE * hid
    return {"bytes": float(b * L), "flops": float(2 * R * n * L)}


def tolerance(case):
    """Prepared inputs and the SwiGLU's output are fp16 (11 bits), sums f32; the hyper-connection forms round to bf16
    (8 bits). About four times the distance measured between the path and exact()."""
    if case["kind"] in ("trunk", "head"):
        return {"rel": 8e-4}
    if case["kind"] == "hc" or case["hc"]:
        return {"rel": 1e-2}
    return {"rel": 1.5e-3}


# ---------------------------------------------------------------------------------------------------- in 64 bits
def _had(v):
    """the normalised Hadamard transform of the last dimension's blocks of 128 (64, 32, 16 where 128 does not divide)"""
    d = v.shape[-1]
    n = next(k for k in (128, 64, 32, 16) if d % k == 0)
    H = torch.ones(1, 1, dtype=torch.float64, device=v.device)
    while H.shape[0] < n:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    return (v.reshape(-1, n) @ (H / math.sqrt(n))).reshape(v.shape)


_slot_cache = {}


def _slots():
    """row and column inside a 16 x 16 tile of the 256 ring slots in order"""
    if not _slot_cache:
        s = torch.arange(256, device="cuda")
        l, j = s >> 3, s & 7
        q = l & 3
        row = torch.stack([2 * q, 2 * q + 1, 2 * q + 8, 2 * q + 9])[j & 3, s]
        _slot_cache["at"] = row * 16 + (l >> 2) + 8 * (j >> 2)
    return _slot_cache["at"]


def _decode(words, K):
    """words int64 [..., 8 K] (a tile's ring as 32-bit words, bits from the highest down) -> f64 [..., 16, 16]: slot
    i's codeword is the 15 bits that end at bit (i + 1) K of the ring; the codebook is the multiplicative one"""
    lo = (torch.arange(256, device="cuda") * K + K - 15) % (256 * K)  # the codeword's first bit
    i0, off = lo >> 5, lo & 31
    w0, w1 = words[..., i0], words[..., (i0 + 1) % (8 * K)]
    two = (w0 << 17) | (w1 >> 15)  # 49 bits from the word's first bit: enough for any 15 that start in it
    cw = (two >> (34 - off)) & 0x7FFF
    r = ((cw * 0xCBAC1FED) & 0x8FFF8FFF) ^ 0x3B603B60
    half = torch.stack([r & 0xFFFF, r >> 16]).to(torch.int32)
    half = torch.where(half >= 32768, half - 65536, half).to(torch.int16).view(torch.float16)
    v = (half[0].float() + half[1].float()).half().double()
    out = torch.empty_like(v)
    out[..., _slots()] = v
    return out.reshape(*v.shape[:-1], 16, 16)


def _words(t):
    """int16 pairs to 32-bit words, as int64"""
    return t.contiguous().view(torch.int32).long() & 0xFFFFFFFF


def _lin64(x, arrays, block=16384):
    t, su, sv = arrays
    K = t.shape[-1] // 16
    xin = _had(x.double() * su.double())
    got = []
    for o in range(0, t.shape[1], block // 16):  # column blocks keep the decoded weights small
        W = _decode(_words(t[:, o:o + block // 16]), K)
        got.append(xin @ W.permute(0, 2, 1, 3).reshape(t.shape[0] * 16, -1))
    return _had(torch.cat(got, 1)) * sv.double()


def _mix64(z):
    """splitmix64 of int64 tensors (wrapping), the recipe of the library's synthetic layers"""
    def shr(v, n):
        return (v >> n) & ((1 << (64 - n)) - 1)

    def c(v):
        return v - (1 << 64) if v >= 1 << 63 else v

    z = z + c(0x9E3779B97F4A7C15)
    z = (z ^ shr(z, 30)) * c(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * c(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def _wrap(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >= 1 << 63 else v


def _syn_words(seed, first, n):
    i = torch.arange(first, first + n, device="cuda", dtype=torch.int64)
    return _mix64(i + _wrap(seed * 0x100000001B3)) & 0xFFFFFFFF


def _syn_gauss(seed, n):
    i = torch.arange(n, device="cuda", dtype=torch.int64)
    h = _mix64((i * _wrap(0xD1B54A32D192ED03)) ^ seed)
    u1 = (((h >> 40) & 0xFFFFFF).float() + 0.5) * (1.0 / 16777216.0)
    u2 = ((h >> 16) & 0xFFFFFF).float() * (1.0 / 16777216.0)
    return torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(6.28318530718 * u2)


def _syn_scale(seed, n):
    m = (1.0 + 0.1 * _syn_gauss(seed, n)).abs()
    neg = _mix64(torch.arange(n, device="cuda", dtype=torch.int64) + (seed + 0x51ED27)) & 1
    return torch.where(neg == 1, -m, m).half().double()


class _Expert:
    """One synthetic expert's three linears: block `at` of the array that fill `wseed` covers"""

    def __init__(self, hid, inter, K, wseed, sseed, at):
        up = lambda v: (v + 255) & ~255  # noqa: E731
        dims = ((hid, inter), (hid, inter), (inter, hid))
        tr = up(hid * inter * K // 8)
        size = 3 * tr + sum(up(2 * i) + up(2 * o) for i, o in dims)
        self.lin = []
        for p, (i, o) in enumerate(dims):
            w = _syn_words(wseed, (at * size + p * tr) // 4, i * o * K // 32).reshape(o // 32, i // 16, 2, 8 * K)
            W = _decode(w, K)  # [pair][k tile][2][16][16]
            self.lin.append((W.permute(1, 3, 0, 2, 4).reshape(i, o), _syn_scale(sseed * 131 + 2 * p, i),
                             _syn_scale(sseed * 131 + 2 * p + 1, o)))

    def __call__(self, x):
        def f(p, v):
            W, su, sv = self.lin[p]
            return _had(_had(v * su) @ W) * sv

        g, u = f(0, x), f(1, x)
        return f(2, torch.nn.functional.silu(g) * u)


def _bf16_64(v):
    """f64 -> the nearest bf16 value, ties to even (through f32 the first rounding could make or break a tie)"""
    m, e = torch.frexp(v)
    return torch.ldexp(torch.round(m * 256) / 256, e)


def _moe64(case, seed, layer, x):
    hid, inter = MOE[case["shape"]]
    ls, K = _moe_seed(seed, layer), case["K"]
    x = x.double()
    sd = torch.tensor(1.0 / math.sqrt(hid), dtype=torch.float32, device="cuda")
    router = (_syn_gauss(ls * 7 + 5, NE * hid) * sd).bfloat16().double().reshape(NE, hid)
    logits = _bf16_64(x @ router.T)  # the router's logits are bf16: ties go to the lower expert
    val, idx = torch.sort(logits, dim=1, descending=True, stable=True)
    wt, idx = torch.softmax(val[:, :TOPK], 1), idx[:, :TOPK]
    y = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        r, k = torch.nonzero(idx == e, as_tuple=True)
        y.index_add_(0, r, _Expert(hid, inter, K, ls * 7 + 1, ls * 100003 + e, e)(x[r]) * wt[r, k][:, None])
    if case["shared"] == "exl3":
        return y + _Expert(hid, inter, case["Ks"], ls * 7 + 3, ls * 100003 + 999983, 0)(x)
    n = inter * hid
    q = _syn_words(ls * 7 + 3, 0, 3 * n // 4)
    q = torch.stack([(q >> s) & 0xFF for s in (0, 8, 16, 24)], 1).reshape(3, n).double()

    def f(p, v, rows, inp):
        sc = ((1.0 + 0.1 * _syn_gauss(ls * 13 + p, n // 128)).abs()
              / (74.0 * torch.sqrt(torch.tensor(float(inp), device="cuda")))).bfloat16().float()
        bi = (-127.5 * sc).bfloat16()
        W = q[p].reshape(-1, 128) * sc.double()[:, None] + bi.double()[:, None]
        return v @ W.reshape(rows, inp).T

    return y + f(2, torch.nn.functional.silu(f(0, x, inter, hid)) * f(1, x, inter, hid), hid, inter)


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "trunk":
        return [[_lin64(x, w) for w in qkv] + [_lin64(a, o)] for qkv, o, x, a in _trunk_arrays(case, g)]
    if kind == "head":
        w = _lin_arrays(g, case["inp"], case["out"], case["K"])
        return [[_lin64(_bf16_values(g, case["rows"], case["inp"]), w)]]
    got = []
    if kind == "hc":
        for d in _hc_arrays(case, g):
            h, R, hid = d["h"].double(), case["rows"], case["hid"]
            inv = 1 / torch.sqrt((h * h).mean(2) + 1e-6)
            hw = h * d["norm"].double().reshape(4, hid)
            xn = hw * inv[:, :, None]
            mix = torch.nn.functional.silu(_lin64(xn.reshape(R, -1), d["down"]) / 4)
            gate = torch.sigmoid(_lin64(mix, d["up"]).reshape(R, 4, hid))
            inj = 2 * torch.sigmoid(xn.reshape(R, -1) @ d["inject"].double().T / 4)
            got.append([mix, torch.cat([inj, inv], 1), (gate * xn).mean(1)])
        return got
    for i, d in enumerate(_moe_inputs(case, g)):
        y = _moe64(case, seed, i, d["x"])
        got.append([y])
        if case["hc"]:
            got[-1].append(d["h"].double() + y[:, None, :] * d["inj"].double()[:, :4, None])
    return got
