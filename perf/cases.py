"""Performance cases of the quantized linear path: what a model runtime asks of libagens_kernels.so, call by call.

Every case goes through the C entry points of include/agens_kernels.h on torch's current stream, with the weights laid
out once by ak_wq_repack_kt as a load path does.  Shapes are the decoder linears this repository's benchmark and tests
use (hidden 5120, MLP 27648, 152064 logits, the 5120 x 6144 linear of the batch-invariance tests); draw() takes other
shapes of the same ranges, odd row counts and token counts among them.

Kinds of case:
  gemv   ak_wq_gemv_kt_multi, default numerics: m tokens through one linear or the three segments q, k, v;
  silu   ak_wq_gemv_kt_silu: the down projection on the merged gate_up output;
  chain  ak_wq_chain_run: the linears of decoder layers and the LM head as one decode step;
  gemm   ak_wq_gemm_kt: prefill from the quantized weights;
  i8     ak_i8_gemv: the INT8 LM head;
  bi     ak_bf16_gemv_bi_ld: a bf16 linear whose rows do not depend on the batch.
`layers` linears of one shape are called one after the other, as the layers of a model are: a model's weights do not fit
the caches, so those of a small linear are not found there either.
"""
import ctypes
import importlib

import torch

DEV = "cuda"
HID, KV, INTER, VOCAB = 5120, 1024, 27648, 152064
_vp, _i, _l = ctypes.c_void_p, ctypes.c_int, ctypes.c_long


class Step(ctypes.Structure):
    """ak_wq_step of include/agens_kernels.h."""
    _fields_ = [("bits", _i), ("m", _i), ("nseg", _i), ("k", _i), ("group", _i), ("bf16w", _i), ("x", _vp),
                ("wt", _vp * 4), ("st", _vp * 4), ("y", _vp * 4), ("n", _i * 4), ("ldy", _i * 4),
                ("independent", _i), ("act", _i)]


_lib = None


def lib():
    global _lib
    if _lib is None:
        k = importlib.import_module("agens-engine_amd").load()
        k.ak_wq_kt_weight_bytes.restype = k.ak_w4_kt_scale_bytes.restype = ctypes.c_size_t
        k.ak_wq_repack_kt.argtypes = [_i, _vp, _vp, _vp, _vp, _i, _i, _i, _vp]
        k.ak_wq_gemv_kt_multi.argtypes = [_i, _vp, _i, _i, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _vp]
        k.ak_wq_gemv_kt_silu.argtypes = [_i, _vp, _i, _vp, _vp, _vp, _i, _i, _i, _i, _vp]
        k.ak_wq_gemm_kt.argtypes = [_i, _vp, _i, _vp, _vp, _vp, _i, _i, _i, _i, _vp]
        k.ak_i8_gemv.argtypes = [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp]
        k.ak_bf16_gemv_bi_ld.argtypes = [_vp, _vp, _vp, _vp, _i, _i, _i, _l, _vp]
        k.ak_wq_chain_create.argtypes = [_vp, _i, _vp]
        k.ak_wq_chain_run.argtypes = [_vp, _vp]
        k.ak_wq_chain_destroy.argtypes = [_vp]
        _lib = k
    return _lib


def stream():
    return torch.cuda.current_stream().cuda_stream


def check(rc):
    if rc:
        raise RuntimeError("libagens_kernels: error %d" % rc)


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one attention output projection for one token: the smallest call of a decode step, bound by latency
        dict(name="o_w4_m1", kind="gemv", bits=4, group=128, m=1, n=HID, n_kv=0, k=HID, layers=1),
        # a decode step of one conversation: two decoder layers (qkv, o, gate_up, SiLU * up and down, W3 with a W4 qkv)
        # and the W4 LM head, each linear reading the one before it
        dict(name="decode_step_m1", kind="chain", m=1, hid=HID, n_kv=KV, inter=INTER, vocab=VOCAB, layers=2,
             bits_qkv=4, bits_o=3, bits_gu=3, bits_down=2, bits_head=4),
        # q, k and v of eight layers for a draft of 8 tokens being verified
        dict(name="qkv_w4_m8", kind="gemv", bits=4, group=128, m=8, n=HID, n_kv=KV, k=HID, layers=8),
        # the MLP's two halves for four conversations: SiLU(gate) * up fused into the long down projection
        dict(name="silu_down_w2_m4", kind="silu", bits=2, group=128, m=4, n=HID, k=INTER, layers=4),
        # the merged gate_up projection, the layer's largest linear, for a batch of 16
        dict(name="gate_up_w3_m16", kind="gemv", bits=3, group=128, m=16, n=2 * INTER, n_kv=0, k=HID, layers=1),
        # the same for 64 tokens: a tree of drafts, or many conversations in one step
        dict(name="gate_up_w3_m64", kind="gemv", bits=3, group=128, m=64, n=2 * INTER, n_kv=0, k=HID, layers=1),
        # the long down projection for an odd number of tokens between the batch sizes
        dict(name="down_w2_m37", kind="gemv", bits=2, group=128, m=37, n=HID, n_kv=0, k=INTER, layers=4),
        # a linear quantized in groups of 64, two tokens
        dict(name="g64_w4_m2", kind="gemv", bits=4, group=64, m=2, n=HID, n_kv=0, k=6144, layers=8),
        # prefill of a 512-token prompt through the merged gate_up projection
        dict(name="prefill_gate_up_w3_t512", kind="gemm", bits=3, group=128, m=512, n=2 * INTER, k=HID, layers=1),
        # prefill of a prompt of 333 tokens through the down projection: ragged token tiles, long k
        dict(name="prefill_down_w2_t333", kind="gemm", bits=2, group=128, m=333, n=HID, k=INTER, layers=1),
        # the INT8 LM head for 4 tokens
        dict(name="i8_head_m4", kind="i8", m=4, n=VOCAB, k=HID, layers=1),
        # a bf16 linear with bias for 16 tokens of a verify step
        dict(name="bf16_bi_m16", kind="bi", m=16, n=HID, k=HID, bias=True, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "gemv", "silu", "chain", "gemm", "gemm", "i8", "bi"])
    bits, group = rng.choice([2, 3, 4]), rng.choice([64, 128, 128, 128])
    k = 128 * _log(rng, 8, 216)
    if kind == "chain":
        hid, inter = 128 * _log(rng, 8, 40), 128 * _log(rng, 16, 216)
        b = [rng.choice([2, 3, 4]) for _ in range(5)]
        return dict(kind=kind, m=rng.choice([1, 1, 2]), hid=hid, n_kv=128 * rng.randint(1, 8), inter=inter,
                    vocab=_log(rng, 8000, VOCAB), layers=rng.randint(1, 2), bits_qkv=b[0], bits_o=b[1], bits_gu=b[2],
                    bits_down=b[3], bits_head=b[4])
    if kind == "i8":
        return dict(kind=kind, m=_log(rng, 1, 16), n=_log(rng, 8000, VOCAB), k=16 * _log(rng, 64, 320), layers=1)
    if kind == "bi":
        return dict(kind=kind, m=_log(rng, 1, 128), n=_log(rng, 48, 8192), k=32 * _log(rng, 32, 256),
                    bias=rng.random() < 0.5, layers=rng.randint(1, 2))
    n = _log(rng, 1000, min(2 * INTER, 2 * INTER * HID // k))
    if kind == "gemm":
        return dict(kind=kind, bits=bits, group=group, m=_log(rng, 129, 512), n=n, k=k, layers=1)
    if kind == "silu":
        return dict(kind=kind, bits=bits, group=128, m=_log(rng, 1, 16), n=min(n, 8192), k=k, layers=rng.randint(1, 2))
    kv = rng.choice([0, 0, n // 5])
    return dict(kind=kind, bits=bits, group=group, m=_log(rng, 1, 128), n=n - 2 * kv, n_kv=kv, k=k, layers=1)


# ------------------------------------------------------------------------------------------------ inputs
# Codes are bell-shaped around zero over the whole range of the bit width, scales positive with the spread of a trained
# linear's, such that outputs have about the size of the inputs; activations are normal with some larger channels.
_FIELD = {4: (0x77777777, 0x11111111), 3: (0x33333333, 0x55555555), 2: (0x11111111, 0x77777777)}
_MEANSQ = {4: 10.6, 3: 2.6, 2: 0.56}  # mean square of the codes below


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _words(g, shape, mask):
    return torch.randint(-2 ** 31, 2 ** 31, shape, dtype=torch.int32, device=DEV, generator=g) & mask


def _container(g, bits, n, k, group, gain=1.0):
    """The int4 container of a linear: words of 8 codes q + 8, and bf16 scales per group."""
    mask, base = _FIELD[bits]
    w = _words(g, (n, k // 8), mask) + _words(g, (n, k // 8), mask) + base  # a triangle symmetric around q = 0
    r = _words(g, (n, k // 8), -1)
    w -= r & (r >> 1) & (r >> 2) & (r >> 3) & 0x11111111  # one code in 16 a step lower: the lowest code occurs too
    s = torch.randn((n, k // group), device=DEV, generator=g).mul_(0.3).exp_()
    s *= gain / (k * _MEANSQ[bits] * 1.2) ** 0.5
    return w, s.to(torch.bfloat16)


def _x(g, m, k):
    x = torch.randn((m, k), device=DEV, generator=g)
    x *= torch.where(torch.rand((1, k), device=DEV, generator=g) < 0.01, 8.0, 1.0)
    return x.to(torch.bfloat16)


def _kt(g, bits, n, k, group, gain=1.0):
    """A linear in the layout the kernels read: (weights, scales)."""
    L = lib()
    w, s = _container(g, bits, n, k, group, gain)
    wt = torch.empty(L.ak_wq_kt_weight_bytes(bits, n, k), dtype=torch.uint8, device=DEV)
    st = torch.empty(L.ak_w4_kt_scale_bytes(n, k, group), dtype=torch.uint8, device=DEV)
    check(L.ak_wq_repack_kt(bits, w.data_ptr(), s.data_ptr(), wt.data_ptr(), st.data_ptr(), n, k, group, stream()))
    return wt, st


def _segments(case):
    kv = case.get("n_kv", 0)
    return [case["n"]] + [kv] * (2 if kv else 0)


def _chain_shapes(c):
    """(name, bits, rows of its segments, k, act, gain) of a decode step's linears in order."""
    steps = []
    for _ in range(c["layers"]):
        steps += [("qkv", c["bits_qkv"], [c["hid"], c["n_kv"], c["n_kv"]], c["hid"], 0, 1.0),
                  ("o", c["bits_o"], [c["hid"]], c["hid"], 0, 1.0),
                  ("gate_up", c["bits_gu"], [2 * c["inter"]], c["hid"], 0, 1.0),
                  ("down", c["bits_down"], [c["hid"]], c["inter"], 1, 2.5)]
    return steps + [("head", c["bits_head"], [c["vocab"]], c["hid"], 0, 1.0)]


class Chain:
    """A chain of decode steps and the buffers it works on."""

    def __init__(self, case, g):
        m, h = case["m"], _x(g, case["m"], case["hid"])
        self.x, self.keep, steps, src = h, [], [], h
        for _, bits, rows, k, act, gain in _chain_shapes(case):
            s = Step(bits=bits, m=m, nseg=len(rows), k=k, group=128, x=src.data_ptr(), act=act)
            ys = []
            for i, n in enumerate(rows):
                wt, st = _kt(g, bits, n, k, 128, gain)
                y = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
                s.wt[i], s.st[i], s.y[i], s.n[i] = wt.data_ptr(), st.data_ptr(), y.data_ptr(), n
                self.keep += [wt, st, y]
                ys.append(y)
            steps.append(s)
            hidden, src = src, ys[0]
        self.logits, self.hidden = src, hidden
        self.steps, self.handle = (Step * len(steps))(*steps), _vp()
        check(lib().ak_wq_chain_create(self.steps, len(steps), ctypes.byref(self.handle)))

    def __del__(self):
        if getattr(self, "handle", None):
            lib().ak_wq_chain_destroy(self.handle)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "chain":
        return {"kind": kind, "chain": Chain(case, g)}
    m, k, n = case["m"], case["k"], case["n"]
    calls = []
    for _ in range(case["layers"]):
        x = _x(g, m, 2 * k if kind == "silu" else k)
        if kind == "i8":
            w = (torch.randn((n, k), device=DEV, generator=g) * 32).round_().clamp_(-127, 127).to(torch.int8)
            s = torch.rand((n,), device=DEV, generator=g) * 1e-3 + 2e-4
            keep = [w, s]
        elif kind == "bi":
            w = (torch.randn((n, k), device=DEV, generator=g) * k ** -0.5).to(torch.bfloat16)
            keep = [w, torch.randn((n,), device=DEV, generator=g).to(torch.bfloat16) if case["bias"] else None]
        else:
            keep = [_kt(g, case["bits"], r, k, case["group"]) for r in _segments(case)]
        ys = [torch.empty((m, r), dtype=torch.bfloat16, device=DEV) for r in _segments(case)]
        args = None
        if kind == "gemv":
            c = len(ys)
            args = ((_vp * c)(*[w.data_ptr() for w, _ in keep]), (_vp * c)(*[s.data_ptr() for _, s in keep]),
                    (_vp * c)(*[y.data_ptr() for y in ys]), (_i * c)(*[y.shape[1] for y in ys]))
        calls.append((x, keep, ys, args))
    return {"kind": kind, "case": case, "calls": calls}


def run(state):
    L, s, kind = lib(), stream(), state["kind"]
    if kind == "chain":
        c = state["chain"]
        check(L.ak_wq_chain_run(c.handle, s))
        return {"logits": c.logits, "hidden": c.hidden}
    case = state["case"]
    m, n, k = case["m"], case["n"], case["k"]
    out = []
    for x, keep, ys, args in state["calls"]:
        if kind == "gemv":
            wt, st, yp, rows = args
            rc = L.ak_wq_gemv_kt_multi(case["bits"], x.data_ptr(), m, len(ys), wt, st, yp, rows, None, k,
                                       case["group"], 0, s)
        elif kind == "i8":
            rc = L.ak_i8_gemv(x.data_ptr(), keep[0].data_ptr(), keep[1].data_ptr(), ys[0].data_ptr(), m, n, k, n, s)
        elif kind == "bi":
            b = keep[1].data_ptr() if keep[1] is not None else None
            rc = L.ak_bf16_gemv_bi_ld(x.data_ptr(), keep[0].data_ptr(), b, ys[0].data_ptr(), m, n, k, n, s)
        else:
            (wt, st), y = keep[0], ys[0]
            f = L.ak_wq_gemv_kt_silu if kind == "silu" else L.ak_wq_gemm_kt
            rc = f(case["bits"], x.data_ptr(), m, wt.data_ptr(), st.data_ptr(), y.data_ptr(), n, n, k, case["group"], s)
        check(rc)
        out.append(ys)
    return out


# ------------------------------------------------------------------------------------------------ what it takes
def _linear_work(bits, m, rows, k, group, x_factor=1):
    n = sum(rows)
    return n * k * bits / 8 + n * (k // group) * 2 + 2 * m * (k * x_factor + n), 2.0 * m * n * k


def work(case):
    kind, b, f = case["kind"], 0.0, 0.0
    if kind == "chain":
        for _, bits, rows, k, act, _ in _chain_shapes(case):
            db, df = _linear_work(bits, case["m"], rows, k, 128, 2 if act else 1)
            b, f = b + db, f + df
        return {"bytes": b, "flops": f}
    m, n, k, layers = case["m"], case["n"], case["k"], case["layers"]
    if kind in ("i8", "bi"):
        per = 1 if kind == "i8" else 2
        return {"bytes": layers * (n * k * per + 4.0 * n + 2 * m * (k + n)), "flops": layers * 2.0 * m * n * k}
    b, f = _linear_work(case["bits"], m, _segments(case), k, case["group"], 2 if kind == "silu" else 1)
    return {"bytes": layers * b, "flops": layers * f}


def tolerance(case):
    """Measured against exact(): one rounding to bf16 is 1.7e-3 in the 2-norm and 2^-8 of a value at most; a decode
    step rounds the output of each of its linears.  About four times that."""
    if case["kind"] == "chain":
        return {"rel": 0.025, "max": 0.15}
    if case["kind"] == "silu":
        return {"rel": 0.008, "max": 0.02}
    return {"rel": 0.007, "max": 0.016}


# ------------------------------------------------------------------------------------------------ 64 bits
def _matmul64(x, w, s, bits, group, round_w=False):
    """x [m][k] times the container's linear transposed, in 64 bits; round_w: weights rounded to bf16(q * scale)."""
    n, k = w.shape[0], w.shape[1] * 8
    out = torch.empty((x.shape[0], n), dtype=torch.float64, device=DEV)
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device=DEV)
    step = max(1, 40_000_000 // k)
    for r in range(0, n, step):
        q = ((w[r:r + step, :, None] >> shifts) & 15).to(torch.float32).sub_(8.0).reshape(-1, k // group, group)
        v = q.mul_(s[r:r + step].to(torch.float32)[:, :, None]).reshape(-1, k)  # exact: 4 times 8 significant bits
        v = v.to(torch.bfloat16) if round_w else v
        out[:, r:r + step] = x @ v.to(torch.float64).t()
    return out


def _silu64(gu):
    g, u = gu.chunk(2, dim=1)
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    g, kind, m = _gen(seed), case["kind"], case["m"]
    if kind == "chain":
        src = _x(g, m, case["hid"]).to(torch.float64)
        for name, bits, rows, k, act, gain in _chain_shapes(case):
            if act:
                src = _silu64(src)
            first = None
            for n in rows:
                w, s = _container(g, bits, n, k, 128, gain)
                if first is None:
                    first = _matmul64(src, w, s, bits, 128)
            hidden, src = src, first
        return {"logits": src, "hidden": hidden}
    out, k, n = [], case["k"], case["n"]
    for _ in range(case["layers"]):
        x = _x(g, m, 2 * k if kind == "silu" else k).to(torch.float64)
        if kind == "i8":
            w = (torch.randn((n, k), device=DEV, generator=g) * 32).round_().clamp_(-127, 127).to(torch.int8)
            s = torch.rand((n,), device=DEV, generator=g) * 1e-3 + 2e-4
            out.append([torch.cat([x @ c.to(torch.float64).t() for c in w.split(8192)], dim=1) * s.to(torch.float64)])
            continue
        if kind == "bi":
            w = (torch.randn((n, k), device=DEV, generator=g) * k ** -0.5).to(torch.bfloat16).to(torch.float64)
            b = torch.randn((n,), device=DEV, generator=g).to(torch.bfloat16).to(torch.float64) if case["bias"] else 0.0
            out.append([x @ w.t() + b])
            continue
        x = _silu64(x).to(torch.bfloat16).to(torch.float64) if kind == "silu" else x  # the activation is bf16
        ys = []
        for r in _segments(case):
            w, s = _container(g, case["bits"], r, k, case["group"])
            ys.append(_matmul64(x, w, s, case["bits"], case["group"], round_w=kind == "gemm"))
        out.append(ys)
    return out
