"""The work this library is timed on, through its C entry points.

A case is one call pattern of a program that serves a dual-precision MoE
model: how many layers it runs, how many tokens each call carries, the layer's
shape, how many experts are hot, the numerics mode, and which entry points it
goes through (`path`: "layer" is llapis_moe_ffn, "fires" the operators of a
graph that keeps them apart: llapis_router_topk, two
llapis_moe_dual_compute fires, llapis_geglu, llapis_moe_combine).

Weights are N(0, 0.02) rounded to each format (IQ2_S: codebook entries, signs
and scales drawn directly), tokens N(0, 1) as after a norm, routing follows a
Zipf(1.1) prior whose most frequent experts are the hot ones, as in bench.py.
Several layers per case keep the weights out of the caches, as a model's other
layers do.
"""
import ctypes as C
import math
import re
from pathlib import Path

import numpy as np
import torch

import llapis_amd as la
from llapis_amd import _lib as L

SHAPE = dict(d_model=2816, n_ff=704, n_expert=128, top_k=8)     # bench.py's layer
PRIOR = 0.5674              # router bias = PRIOR * log(Zipf prior): about 85 % of the picks are hot at K = 57 of 128
I32 = 26                    # ggml's type tag of an int32 tensor


def _case(name, tokens, layers=1, k_slots=57, path="layer", mode="cpu", scales=False, x_router=False, **shape):
    c = dict(SHAPE, name=name, tokens=tokens, layers=layers, k_slots=k_slots, path=path, mode=mode, scales=scales,
             x_router=x_router)
    c.update(shape)
    return c


def listed():
    return [
        # decode of one token by a model whose experts are all cold: one layer, the smallest call there is
        _case("token_cold", 1, k_slots=0),
        # a token through the layers of a model that fits whole in the hot formats
        _case("token_hot", 1, layers=16, k_slots=128),
        # ordinary decode, mixed precision, per-expert scales and the router on its own input
        _case("token_dual", 1, layers=16, scales=True, x_router=True),
        # a three-deep speculative verify: the headline of bench.py
        _case("verify4_dual", 4, layers=8),
        # a shorter verify in the ggml-cuda numerics
        _case("verify3_q81", 3, layers=8, mode="q8_1"),
        # a verify by a graph that keeps the operators apart
        _case("fires4_dual", 4, layers=8, path="fires", scales=True),
        # a server's decode batch: one token from each of a dozen users
        _case("batch12_dual", 12, layers=4),
        # a larger batch in the ggml-cuda numerics
        _case("batch48_q81", 48, layers=2, mode="q8_1"),
        # the odd end of a prompt, on a smaller layer
        _case("tail173_dual", 173, layers=2, k_slots=40, d_model=2048, n_ff=768, n_expert=96, top_k=6, scales=True),
        # a prompt chunk, mixed precision: bench.py's prefill
        _case("chunk512_dual", 512),
        # the same in the ggml-cuda numerics
        _case("chunk512_q81", 512, mode="q8_1"),
        # a long prompt in one call, every expert at the hot precision
        _case("prompt1900_hot", 1900, k_slots=128),
    ]


def draw(rng):
    n_expert = 8 * rng.randint(4, 32)
    top_k = rng.randint(2, 10)
    d_model = 256 * rng.randint(4, 12)
    n_ff = 64 * rng.randint(4, 16)
    path = "fires" if rng.random() < 0.15 else "layer"
    most = 4 if path == "fires" else 2048
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(most + 0.49)))))
    if path == "fires":
        tokens = min(tokens, 32 // top_k)
    else:                       # no more arithmetic than the largest listed case
        tokens = min(tokens, int(1900 * 8 * 704 * 2816 / (top_k * n_ff * d_model)))
    tokens = max(tokens, 1)
    layers = rng.randint(1, 8) if tokens <= 4 else rng.randint(1, 3) if tokens <= 64 else 1
    k_slots = rng.choice([0, n_expert, rng.randint(1, n_expert), rng.randint(1, n_expert)])
    mode = "q8_1" if rng.random() < 0.3 else "cpu"
    return dict(tokens=tokens, layers=layers, k_slots=k_slots, path=path, mode=mode, scales=rng.random() < 0.4,
                x_router=path == "layer" and rng.random() < 0.4, d_model=d_model, n_ff=n_ff, n_expert=n_expert,
                top_k=top_k)


# ---------------------------------------------------------------- formats

IQ4_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _iq2_codebook(device):
    """The IQ2_S codebook [1024][8] (data of the format) from the 16-bit codes
    the library is built with: element i of an entry is bits 2 i, 2 i + 1."""
    text = (Path(la.__file__).resolve().parent / "csrc" / "iq2s_grid.inc").read_text()
    codes = torch.tensor([int(v, 16) for v in re.findall(r"\b0x([0-9a-f]{4})\b", text)], device=device)
    assert codes.numel() == 1024
    level = (codes[:, None] >> (2 * torch.arange(8, device=device))) & 3
    return torch.tensor([8.0, 25.0, 43.0, 0.0], dtype=torch.float64, device=device)[level]


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _to_q4_k(w):                # [rows, n] float32 -> [rows, n / 256 * 144] bytes
    x = w.reshape(-1, 8, 32)
    lo = x.amin(2).clamp(max=0)
    scale = (x.amax(2) - lo) / 15
    d, m = scale.amax(1, True) / 63, (-lo).amax(1, True) / 63
    sc = (scale / d).round().clamp(1, 63)
    mn = (-lo / m.clamp(min=1e-30)).round().clamp(0, 63)
    dh, mh = d.half().float(), m.half().float()
    q = ((x + (mh * mn)[..., None]) / (dh * sc)[..., None]).round().clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    head = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                      (sc[:, 4:] & 15) | (mn[:, 4:] << 4)], 1)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    return torch.cat([_half_bytes(d[:, 0]), _half_bytes(m[:, 0]), head, qs], 1).reshape(w.shape[0], -1)


def _to_q5_0(w):
    x = w.reshape(-1, 32)
    d = x.gather(1, x.abs().argmax(1, True)) / -16
    q = (x / d.half().float() + 16).round().clamp(0, 31).to(torch.int64)
    qh = ((q >> 4) << torch.arange(32, device=w.device)).sum(1)
    qh = ((qh[:, None] >> (8 * torch.arange(4, device=w.device))) & 255).to(torch.uint8)
    qs = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
    return torch.cat([_half_bytes(d[:, 0]), qh, qs], 1).reshape(w.shape[0], -1)


def _to_iq4_nl(w):
    x = w.reshape(-1, 32)
    d = x.abs().amax(1, True) / 127
    lev = torch.tensor(IQ4_LEVELS, dtype=torch.float32, device=w.device)
    q = torch.bucketize(x / d.half().float(), (lev[1:] + lev[:-1]) / 2).to(torch.uint8)
    return torch.cat([_half_bytes(d[:, 0]), q[:, :16] | (q[:, 16:] << 4)], 1).reshape(w.shape[0], -1)


def _draw_iq2_s(rows, n, gen, device):
    """Blocks whose values are spread as N(0, 0.02)'s are: any codebook entry
    and signs, sub-block scales in the upper half of their range."""
    blocks = rows * n // 256
    b = torch.randint(0, 256, (blocks, 82), dtype=torch.uint8, device=device, generator=gen)
    d = 2.6e-4 * (0.9 + 0.2 * torch.rand(blocks, device=device, generator=gen))
    b[:, :2] = _half_bytes(d)
    b[:, 74:] = b[:, 74:] | 0x88
    return b.reshape(rows, -1)


def _values(kind, b, n, device, codebook=None):
    """Bytes [rows, .] of a format -> float64 values [rows, n]."""
    rows = b.shape[0]
    half = lambda v: v.contiguous().view(torch.float16).double()
    if kind == "q4_k":
        b = b.reshape(-1, 144)
        s = b[:, 4:16].to(torch.int64)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (half(b[:, :2]) * sc)[..., None] * q - (half(b[:, 2:4]) * mn)[..., None]
    elif kind == "iq2_s":
        b = b.reshape(-1, 82)
        i = torch.arange(32, device=device)
        hi = (b[:, 66:74].to(torch.int64)[:, i // 4] >> (2 * (i % 4))) & 3
        g = codebook[b[:, 2:34].to(torch.int64) | (hi << 8)]                             # [., 32, 8]
        sg = (b[:, 34:66].to(torch.int64)[..., None] >> torch.arange(8, device=device)) & 1
        ls = b[:, 74:82].to(torch.int64)[:, i // 4] >> (4 * ((i // 2) % 2)) & 15
        v = g * (1 - 2 * sg) * (half(b[:, :2]) * (ls.double() * 2 + 1) / 8)[..., None]
    else:
        b = b.reshape(-1, 22 if kind == "q5_0" else 18)
        qs = b[:, -16:]
        q = torch.cat([qs & 15, qs >> 4], 1).to(torch.int64)
        if kind == "q5_0":
            i = torch.arange(32, device=device)
            q = q | (((b[:, 2:6].to(torch.int64)[:, i // 8] >> (i % 8)) & 1) << 4)
            v = (q - 16).double()
        else:
            v = torch.tensor(IQ4_LEVELS, dtype=torch.float64, device=device)[q]
        v = v * half(b[:, :2])
    return v.reshape(rows, n)


# ------------------------------------------------------------------ inputs

def _inputs(case, seed):
    """Weights, tokens and placement of a case, on the GPU, from the seed alone."""
    dev = torch.device("cuda")
    gen = torch.Generator(dev)
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    D, F, E, K = (case[k] for k in ("d_model", "n_ff", "n_expert", "top_k"))
    T, NL, KS = case["tokens"], case["layers"], case["k_slots"]
    perm = rng.permutation(E)
    prior = np.empty(E)
    prior[perm] = 1.0 / np.arange(1, E + 1) ** 1.1
    s = dict(hot=perm[:KS].astype(np.int64))
    s["router_w"] = 0.02 * torch.randn(E, D, device=dev, generator=gen)
    s["router_b"] = torch.tensor(PRIOR * np.log(prior / prior.sum()), dtype=torch.float32, device=dev)
    normal = lambda r, n: 0.02 * torch.randn(r, n, device=dev, generator=gen)
    at_once = max(1, 1 << 27 >> (2 * F * D).bit_length())      # experts rounded at once
    pool = lambda count, f: torch.cat([f(min(at_once, count - e)) for e in range(0, count, at_once)]) \
        if count else torch.zeros(1, 256, dtype=torch.uint8, device=dev)
    s["hot_gu"] = pool(KS, lambda n: _to_q4_k(normal(n * 2 * F, D)).reshape(n, -1))
    s["hot_dn"] = pool(KS, lambda n: _to_q5_0(normal(n * D, F)).reshape(n, -1))
    s["cold_gu"] = pool(E, lambda n: _draw_iq2_s(n * 2 * F, D, gen, dev).reshape(n, -1))
    s["cold_dn"] = pool(E, lambda n: _to_iq4_nl(normal(n * D, F)).reshape(n, -1))
    scale = lambda n: 1 + 0.25 * torch.randn(n, device=dev, generator=gen)
    s["s_hot"], s["s_cold"] = (scale(max(KS, 1)), scale(E)) if case["scales"] else (None, None)
    # tokens; one whose routing hangs on the last bits of its logits is drawn
    # again, so that every correct router agrees about it
    x = torch.randn(NL, T, D, device=dev, generator=gen)
    xr = torch.randn(NL, T, D, device=dev, generator=gen) if case["x_router"] else x
    w64, b64 = s["router_w"].double(), s["router_b"].double()
    for _ in range(8):
        top = (xr.double() @ w64.T + b64).topk(min(K + 1, E), 2).values
        close = (top[..., :-1] - top[..., 1:]).amin(2) < 2e-5
        if not bool(close.any()):
            break
        xr[close] = torch.randn(int(close.sum()), D, device=dev, generator=gen)
    s["x"], s["xr"] = x, xr
    return s


def _layer_inputs(s, i):
    """Layer i holds the same experts in another order (expert e of layer 0 is
    its expert e + i), in buffers of its own."""
    E = s["router_w"].shape[0]
    v = {k: s[k].roll(i, 0).contiguous() if i else s[k] for k in ("router_w", "router_b", "cold_gu", "cold_dn")}
    v["s_cold"] = None if s["s_cold"] is None else s["s_cold"].roll(i, 0).contiguous()
    v.update({k: s[k].clone() if i else s[k] for k in ("hot_gu", "hot_dn")}, s_hot=s["s_hot"])
    v["hot"] = (s["hot"] + i) % E
    return v


def _mirrors(hot, n_expert, device):
    exp_slot = np.full(n_expert, -1, np.int32)
    exp_slot[hot] = np.arange(len(hot), dtype=np.int32)
    slot_exp = np.full(max(len(hot), 1), -1, np.int32)
    slot_exp[:len(hot)] = hot
    state = np.full(max(len(hot), 1), la.SLOT_READY if len(hot) else 0, np.int32)
    return [torch.from_numpy(a).to(device) for a in (exp_slot, slot_exp, state)]


def _tensor(kind, ne, data, row_bytes):
    t = L.LlapisTensor()
    t.type = kind
    for i in range(4):
        t.ne[i] = ne[i] if i < len(ne) else 1
    t.nb[0], t.nb[1] = 4, row_bytes
    t.nb[2] = t.nb[1] * t.ne[1]
    t.nb[3] = t.nb[2] * t.ne[2]
    t.data = data.data_ptr()
    return t


def _fire(case, kind, v, cur, ids, dst, keep):
    """The op of one fire, as a graph holds it."""
    D, F, E, K, T = (case[k] for k in ("d_model", "n_ff", "n_expert", "top_k", "tokens"))
    d_in, d_out = (D, 2 * F) if kind == 0 else (F, D)
    ht, ct = (la.Q4_K, la.IQ2_S) if kind == 0 else (la.Q5_0, la.IQ4_NL)
    hot, cold = (v["hot_gu"], v["cold_gu"]) if kind == 0 else (v["hot_dn"], v["cold_dn"])
    slots = max(case["k_slots"], 1)
    src = [_tensor(la.F32, [d_in, 1 if kind == 0 else K, T], cur, 4 * d_in),
           _tensor(I32, [K, T], ids, 4 * K),
           _tensor(ht, [d_in, d_out, slots], hot, la.row_size(ht, d_in)),
           _tensor(ct, [d_in, d_out, E], cold, la.row_size(ct, d_in)),
           _tensor(I32, [E], v["exp_slot"], 4 * E), _tensor(I32, [slots], v["slot_exp"], 4 * slots),
           _tensor(I32, [slots], v["slot_state"], 4 * slots)]
    op = L.LlapisMoeDualOp()
    if kind == 1 and v["s_hot"] is not None:
        src += [_tensor(la.F32, [slots], v["s_hot"], 4 * slots), _tensor(la.F32, [E], v["s_cold"], 4 * E)]
    out = _tensor(la.F32, [d_out, K, T], dst, 4 * d_out)
    for i, t in enumerate(src):
        op.src[i] = C.pointer(t)
    for i, p in enumerate([kind, K, 0, ct, E, 0, 0, 0, 0, 0]):
        op.op_params[i] = p
    op.dst = C.pointer(out)
    keep += src + [out]
    return op


def prepare(case, seed):
    s = _inputs(case, seed)
    lib, dev = la.lib(), s["x"].device
    D, F, E, K = (case[k] for k in ("d_model", "n_ff", "n_expert", "top_k"))
    T, NL, KS = case["tokens"], case["layers"], case["k_slots"]
    act, gelu = (la.ACT_CPU, la.GELU_TABLE) if case["mode"] == "cpu" else (la.ACT_Q8_1, la.GELU_TANH)
    new = lambda *n, t=torch.float32: torch.zeros(NL, *n, dtype=t, device=dev)
    st = dict(lib=lib, case=case, modes=(act, gelu), keep=[s], calls=[], out=new(T, D), w=new(T, K),
              ids=new(T, K, t=torch.int32))
    if case["path"] == "fires":
        st.update(probs=new(T, E), gu=new(T, K, 2 * F), act=new(T * K, F), dn=new(T, K, D))
    for i in range(NL):
        v = _layer_inputs(s, i)
        v["exp_slot"], v["slot_exp"], v["slot_state"] = _mirrors(v["hot"], E, dev)
        st["keep"].append(v)
        p = lambda t: None if t is None else t.data_ptr()
        x, xr, out, ids, w = (t[i] for t in (s["x"], s["xr"], st["out"], st["ids"], st["w"]))
        if case["path"] == "layer":
            desc = L.LlapisMoeLayer(D, F, E, K, KS, la.Q4_K, la.Q5_0, la.IQ2_S, la.IQ4_NL, act, gelu,
                                    *(p(v[k]) for k in ("router_w", "router_b", "hot_gu", "hot_dn", "cold_gu", "cold_dn",
                                                        "exp_slot", "slot_exp", "slot_state", "s_hot", "s_cold")),
                                    None, None)
            if "ws" not in st:      # one workspace serves the layers, which run one after another
                st["ws"] = torch.zeros(lib.llapis_moe_ffn_workspace_size(C.byref(desc), T), dtype=torch.uint8, device=dev)
            st["calls"].append((C.byref(desc), x.data_ptr(), p(xr) if case["x_router"] else None, T, out.data_ptr(),
                                ids.data_ptr(), w.data_ptr(), st["ws"].data_ptr(), st["ws"].numel()))
        else:
            gu, act_, dn, probs = (st[k][i] for k in ("gu", "act", "dn", "probs"))
            ops = [_fire(case, 0, v, x, ids, gu, st["keep"]), _fire(case, 1, v, act_, ids, dn, st["keep"])]
            if "ws" not in st:
                n = max(lib.llapis_moe_dual_workspace_size(C.byref(o)) for o in ops)
                st["ws"] = torch.zeros(n, dtype=torch.uint8, device=dev)
            ws = (st["ws"].data_ptr(), st["ws"].numel())
            st["calls"].append((
                (xr.data_ptr(), T, p(v["router_w"]), p(v["router_b"]), D, E, K, ids.data_ptr(), w.data_ptr(), probs.data_ptr()),
                (C.byref(ops[0]),) + ws, (gu.data_ptr(), F, T * K, act_.data_ptr(), gelu), (C.byref(ops[1]),) + ws,
                (dn.data_ptr(), w.data_ptr(), T, K, D, out.data_ptr())))
    return st


def run(state):
    lib, stream = state["lib"], torch.cuda.current_stream().cuda_stream
    rc = 0
    if state["case"]["path"] == "layer":
        for call in state["calls"]:
            rc |= lib.llapis_moe_ffn(*call, stream)
    else:
        lib.llapis_set_modes(*state["modes"])
        for router, up, geglu, down, comb in state["calls"]:
            rc |= lib.llapis_router_topk(*router, stream)
            rc |= lib.llapis_moe_dual_compute(*up, stream)
            rc |= lib.llapis_geglu(*geglu, stream)
            rc |= lib.llapis_moe_dual_compute(*down, stream)
            rc |= lib.llapis_moe_combine(*comb, stream)
    if rc:
        raise RuntimeError(lib.llapis_last_error().decode())
    names = ("out", "ids", "w") + (("gu", "act", "dn") if state["case"]["path"] == "fires" else ())
    return {k: state[k] for k in names}


# ------------------------------------------------------------------- bounds

def _distinct(case):
    """Expected distinct hot and cold experts a call's tokens are routed to."""
    E, K, T = case["n_expert"], case["top_k"], case["tokens"]
    rng = np.random.default_rng(1)
    prior = 1.0 / np.arange(1, E + 1) ** 1.1
    z = rng.standard_normal((4096, E)) * 0.02 * math.sqrt(case["d_model"]) + PRIOR * np.log(prior / prior.sum())
    p = np.bincount(np.argpartition(-z, K - 1, 1)[:, :K].ravel(), minlength=E) / 4096
    seen = 1 - (1 - p) ** T
    return float(seen[:case["k_slots"]].sum()), float(seen[case["k_slots"]:].sum())


def work(case):
    D, F, E, K = (case[k] for k in ("d_model", "n_ff", "n_expert", "top_k"))
    T, NL = case["tokens"], case["layers"]
    size = lambda t, n, rows: la.row_size(t, n) * rows
    hot, cold = _distinct(case)
    bytes_ = hot * (size(la.Q4_K, D, 2 * F) + size(la.Q5_0, F, D)) + cold * (size(la.IQ2_S, D, 2 * F) + size(la.IQ4_NL, F, D))
    bytes_ += E * D * 4 + T * D * (12 if case["x_router"] else 8) + T * K * 8
    if case["path"] == "fires":         # each operator's output goes to memory and is read by the next
        bytes_ += 2 * 4 * T * (E + K * (2 * F + F + D))
    return {"bytes": NL * bytes_, "flops": NL * 2 * (T * K * 3 * F * D + T * E * D)}


def tolerance(case):
    # The sums are in 32 bits, but the activations between gate_up and down are
    # rounded to 8: a sum that differs in its last bits moves a few of them by
    # one step, 1/127 of a block's largest (about 3 times its root mean square).
    # Measured against exact(): 1e-7 without such a value, up to 2e-4 with
    # them; a few of one call's at the smallest sizes weigh more.
    return {"rel": 5e-4 + 4 * 3 / (127 * math.sqrt(case["tokens"] * case["top_k"] * case["n_ff"]))}


# -------------------------------------------------------- the same in 64 bits

def _q8_k(x):                   # [n, D] float32 -> rounded values, float64 (integers times a 32-bit scale per 256)
    b = x.reshape(-1, 256)
    inv = b.new_tensor([-127.0]) / b.gather(1, b.abs().argmax(1, True))     # tensors: torch multiplies by a number's inverse
    q = (inv * b).round().clamp(max=127)
    return (q.double() * (b.new_tensor([1.0]) / inv).double()).reshape(x.shape)


def _q8_32(x, away):            # per 32 values, the scale kept in 16 bits (q8_0; away from zero: q8_1)
    b = x.float().reshape(-1, 32)
    top, n127 = b.abs().amax(1, True), b.new_tensor([127.0])
    d = top / n127
    if away:
        v = torch.where(top > 0, b / d, torch.zeros_like(b))
        q = torch.sign(v) * (v.abs() + 0.5).floor()
    else:
        q = (b * torch.where(top > 0, n127 / top, torch.zeros_like(top))).round()
    return (q.double() * d.half().double()).reshape(x.shape)


def _geglu(g, u, table):
    gelu = lambda v: 0.5 * v * (1 + torch.tanh(0.79788456080286535588 * v * (1 + 0.044715 * v * v)))
    if not table:
        return gelu(g) * u
    y = gelu(g.half().double()).half().double()                # the CPU path looks gelu up at 16 bits
    return torch.where(g <= -10, torch.zeros_like(g), torch.where(g >= 10, g, y)) * u


def exact(case, seed):
    s = _inputs(case, seed)
    dev = s["x"].device
    D, F, E, K = (case[k] for k in ("d_model", "n_ff", "n_expert", "top_k"))
    T, cpu = case["tokens"], case["mode"] == "cpu"
    # up to four tokens the ggml-cuda numerics truncate some sums to integers
    # on the way, which has no value in 64 bits
    whole = cpu or (case["path"] == "layer" and T > 4)
    book = _iq2_codebook(dev)
    res = {k: [] for k in ("out", "ids", "w", "gu", "act", "dn")}
    for i in range(case["layers"]):
        hot = {int(e): k for k, e in enumerate((s["hot"] + i) % E)}
        p = (s["xr"][i].double() @ s["router_w"].roll(i, 0).double().T + s["router_b"].roll(i, 0).double()).softmax(1)
        top = p.topk(K, 1)
        ids, w = top.indices, top.values / top.values.sum(1, True).clamp(min=6.103515625e-5)
        res["ids"].append(ids.int())
        res["w"].append(w)
        if not whole:
            continue
        xq = _q8_k(s["x"][i]) if cpu else _q8_32(s["x"][i], True)
        gu, act, dn = (torch.zeros(T, K, n, dtype=torch.float64, device=dev) for n in (2 * F, F, D))
        for e in ids.unique().tolist():
            t, k = (ids == e).nonzero(as_tuple=True)
            sc = 1.0
            if e in hot:
                wg = _values("q4_k", s["hot_gu"][hot[e]].reshape(2 * F, -1), D, dev)
                wd = _values("q5_0", s["hot_dn"][hot[e]].reshape(D, -1), F, dev)
                sc = 1.0 if s["s_hot"] is None else s["s_hot"][hot[e]].double()
            else:
                c = (e - i) % E
                wg = _values("iq2_s", s["cold_gu"][c].reshape(2 * F, -1), D, dev, book)
                wd = _values("iq4_nl", s["cold_dn"][c].reshape(D, -1), F, dev)
                sc = 1.0 if s["s_cold"] is None else s["s_cold"][c].double()
            y = xq[t] @ wg.T
            a = _geglu(y[:, :F], y[:, F:], cpu)
            gu[t, k], act[t, k] = y, a
            dn[t, k] = sc * (_q8_32(a, not cpu) @ wd.T)
        for name, v in (("gu", gu), ("act", act.reshape(T * K, F)), ("dn", dn), ("out", (dn * w[..., None]).sum(1))):
            res[name].append(v)
    names = ("out", "ids", "w") + (("gu", "act", "dn") if case["path"] == "fires" else ())
    return {k: torch.stack(res[k]) if res[k] else None for k in names}
