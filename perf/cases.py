"""The work that users of this framework have it do, as cases that can be timed and compared.

A speech encoder's five-value linears are called alone (fp32 rows in, as the engine's p2_sgemm_fvb does), inside a
device-resident feed-forward, block or 24-block window, and through the blas.h drop-in on host arrays. Frames per call
range from a word (M = 9: 0.7 s at 80 ms a frame) over a 3 s utterance (38), 10 s (125), one 30 s window (375) and the
longest window (35 s: 438) to sixteen stacked windows (6000). K and N are the encoder's own (1024, 2048, 3072, 4096),
and in drawn cases also ragged ones the entry points take.

Every case runs through phonon-2-c_amd/p2gemm.py (the ctypes binding of include/p2hip.h) or libphonon2_gemm.so
(include/p2_blas.h); prepare() holds what a program keeps: weights on the device, workspace, output buffers, a stream
and, for the window, its captured graph.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch   # before the binding, so that the process holds one HIP runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "phonon-2-c_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import p2gemm as P  # noqa: E402

D, FF, H, DH = 1024, 4096, 8, 128
SHAPES = ((1024, 4096), (4096, 1024), (1024, 3072), (1024, 2048), (1024, 1024))


def listed():
    return [
        # the smallest call: a word's frames through a square linear, where launches and latency are all there is
        {"name": "linear_int8w_m9", "kind": "linear", "mode": "int8w", "M": 9, "K": 1024, "N": 1024},
        # a 3 s utterance's feed-forward down-projection: a long contraction with few rows
        {"name": "linear_int8w_m38_down", "kind": "linear", "mode": "int8w", "M": 38, "K": 4096, "N": 1024},
        # sixteen stacked windows through the up-projection: the throughput case
        {"name": "linear_int8w_m6000_up", "kind": "linear", "mode": "int8w", "M": 6000, "K": 1024, "N": 4096},
        # four ragged windows' qkv with exact weights and int8 rows (the two-plane mode)
        {"name": "linear_int8_m1501_qkv", "kind": "linear", "mode": "int8", "M": 1501, "K": 1024, "N": 3072},
        # one 30 s window's up-projection in the --exact mode
        {"name": "linear_exact_m375_up", "kind": "linear", "mode": "exact", "M": 375, "K": 1024, "N": 4096},
        # sixteen windows' down-projection in the --exact mode
        {"name": "linear_exact_m6000_down", "kind": "linear", "mode": "exact", "M": 6000, "K": 4096, "N": 1024},
        # one window's subsampling output linear, an int8 table with one scale per column
        {"name": "table_int8w_m375", "kind": "table", "mode": "int8w", "M": 375, "K": 4096, "N": 1024},
        # sixteen windows' feed-forward half step on the device (norm, up with SiLU, quantise, down onto the residual)
        {"name": "feed_forward_int8w_m6000", "kind": "feed_forward", "mode": "int8w", "T": 6000},
        # the longest window's relative-position attention, all heads
        {"name": "attention_t438", "kind": "attention", "T": 438},
        # one conformer block of a 10 s clip in the --exact mode, launched call by call
        {"name": "block_exact_t125", "kind": "block", "mode": "exact", "T": 125},
        # a whole 30 s window: 24 blocks replayed from one graph, as a serving loop runs them
        {"name": "window_int8w_t375", "kind": "window", "mode": "int8w", "T": 375, "blocks": 24},
        # the engine's own call on host arrays: one window's up-projection through the blas.h drop-in
        {"name": "host_linear_m375", "kind": "host", "M": 375, "K": 1024, "N": 4096},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "table", "feed_forward", "attention", "block", "window",
                       "host"))
    mode = rng.choice(("int8w", "int8w", "int8", "exact"))
    if kind in ("linear", "host"):
        M = _log_int(rng, 1, 6000 if kind == "linear" else 1500)
        if rng.random() < 0.75:
            K, N = rng.choice(SHAPES)
        else:
            K, N = 4 * _log_int(rng, 64, 1024), 16 * _log_int(rng, 16, 256)
        c = {"kind": kind, "M": M, "K": K, "N": N}
        return dict(c, mode=mode) if kind == "linear" else c
    if kind == "table":
        K, N = rng.choice(((4096, 1024), (1024, 640)))
        return {"kind": kind, "mode": rng.choice(("int8w", "exact")), "M": _log_int(rng, 9, 1500), "K": K, "N": N}
    if kind == "feed_forward":
        return {"kind": kind, "mode": rng.choice(("int8w", "int8")), "T": _log_int(rng, 9, 6000)}
    if kind == "attention":
        return {"kind": kind, "T": _log_int(rng, 9, 768)}
    if kind == "block":
        return {"kind": kind, "mode": mode, "T": _log_int(rng, 9, 438)}
    return {"kind": kind, "mode": rng.choice(("int8w", "int8w", "exact")), "T": _log_int(rng, 38, 375),
            "blocks": rng.choice((6, 12, 24))}


# ── inputs, from the seed alone ─────────────────────────────────────────────────────────────────────────────────

def _gen(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _rows(g, M, K):
    """Activations: unit normals with one value in a thousand twenty times as large."""
    a = torch.randn(M, K, generator=g, device=g.device)
    return a * torch.where(torch.rand(M, K, generator=g, device=g.device) < 0.001, 20.0, 1.0)


def _planes(g, K, N):
    """A five-value weight: codes 0 (0.4), ±lo (0.4), ±hi (0.2), lo ~ U(0.005, 0.02), hi = lo·U(2, 4), both fp16
    values, packed as the reference stores them (signs [K][N/4], flags [K][N/8])."""
    dev = g.device
    u = torch.rand(K, N, generator=g, device=dev)
    code = torch.where(u < 0.3, 0, torch.where(u < 0.7, 1, 2)).to(torch.uint8)
    v = torch.rand(K, N, generator=g, device=dev)
    flag = ((code != 1) & (v < 1.0 / 3.0)).to(torch.uint8)
    two = torch.arange(4, device=dev, dtype=torch.uint8) * 2
    one = torch.arange(8, device=dev, dtype=torch.uint8)
    signs = (code.view(K, N // 4, 4) << two).sum(-1, dtype=torch.int32).to(torch.uint8).contiguous()
    # N % 16 == 0, so every plane row is whole bytes
    flags = (flag.view(K, N // 8, 8) << one).sum(-1, dtype=torch.int32).to(torch.uint8).contiguous()
    lo = (0.005 + 0.015 * torch.rand(N, generator=g, device=dev)).half().float()
    hi = (lo * (2.0 + 2.0 * torch.rand(N, generator=g, device=dev))).half().float()
    return {"code": code, "flag": flag, "signs": signs, "flags": flags, "lo": lo, "hi": hi}


def _vec(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=g.device) * scale


def _norm(g):
    return 0.5 + torch.rand(D, generator=g, device=g.device), 0.4 * torch.rand(D, generator=g, device=g.device) - 0.2


def _block_inputs(g):
    """One conformer block's planes and vectors, keyed as P2hBlock names them. The linears that write onto the residual
    rows have an eighth of the others' values: in a trained encoder a block changes its rows, it does not replace them
    (and rows that are replaced 48 times over carry every rounding on to the end)."""
    b = {name: _planes(g, K, N) for name, (K, N) in P.BLOCK_LINEARS.items()}
    for name in ("ff1_l2", "out", "pw2", "ff2_l2"):
        b[name]["lo"], b[name]["hi"] = b[name]["lo"] / 8, b[name]["hi"] / 8
    for n in ("norm_ff1", "norm_sa", "norm_conv", "norm_ff2", "norm_out"):
        b[n + "_w"], b[n + "_b"] = _norm(g)
    b["bias_u"], b["bias_v"] = _vec(g, D, scale=0.1), _vec(g, D, scale=0.1)
    b["dw_w"], b["dw_b"] = _vec(g, D * P.CONV_K, scale=0.3), _vec(g, D, scale=0.1)
    return b


def _positions(T, device):
    """The sinusoidal table of positions T − 1 .. −(T − 1), [2T − 1][1024]."""
    pos = torch.arange(T - 1, -T, -1, device=device, dtype=torch.float64)[:, None]
    div = torch.exp(torch.arange(0, D, 2, device=device, dtype=torch.float64) * (-math.log(10000.0) / D))
    pe = torch.empty(2 * T - 1, D, device=device, dtype=torch.float64)
    pe[:, 0::2], pe[:, 1::2] = torch.sin(pos * div), torch.cos(pos * div)
    return pe.float()


def _inputs(case, seed, device):
    """What a case's computation is a function of, as torch tensors."""
    g, k = _gen(seed, device), case["kind"]
    if k in ("linear", "host"):
        return {"a": _rows(g, case["M"], case["K"]), "w": _planes(g, case["K"], case["N"])}
    if k == "table":
        a = _rows(g, case["M"], case["K"])
        b = torch.clamp(torch.round(_vec(g, case["K"], case["N"], scale=40.0)), -127, 127).to(torch.int8)
        return {"a": a, "b": b, "s": 0.0002 + 0.0006 * torch.rand(case["N"], generator=g, device=device)}
    T = case["T"]
    if k == "feed_forward":
        gamma, beta = _norm(g)
        return {"x": _rows(g, T, D), "gamma": gamma, "beta": beta, "l1": _planes(g, D, FF), "l2": _planes(g, FF, D)}
    if k == "attention":
        return {"qkv": _vec(g, T, 3 * D), "bu": _vec(g, D, scale=0.1), "bv": _vec(g, D, scale=0.1),
                "p": _vec(g, 2 * T - 1, D)}
    n = case["blocks"] if k == "window" else 1
    return {"x": _rows(g, T, D), "pe": _positions(T, device), "blocks": [_block_inputs(g) for _ in range(n)]}


# ── what a program holds ────────────────────────────────────────────────────────────────────────────────────────

_stream = None


def _the_stream():
    global _stream
    if _stream is None:
        P.init()
        _stream = P.Stream()
    return _stream


def _weight(p, K, N):
    return P.FvWeight.wrap(p["signs"].data_ptr(), p["flags"].data_ptr(), p["lo"].data_ptr(), p["hi"].data_ptr(), K, N,
                           keep=(p["lo"], p["hi"]))


def _workspace(nbytes):
    return P.Workspace(nbytes)


def _dev_block(b):
    """P.Block over device tensors: the weights wrapped, the vectors used where they lie."""
    blk = P.Block.__new__(P.Block)
    blk._keep = {f: _weight(b[f], *P.BLOCK_LINEARS[f]) if f in P.BLOCK_LINEARS else b[f].contiguous()
                 for f in P.BLOCK_FIELDS}
    blk.c = P._P2hBlock(**{f: v.ptr if f in P.BLOCK_LINEARS else v.data_ptr() for f, v in blk._keep.items()})
    return blk


def prepare(case, seed):
    k = case["kind"]
    st = {"case": dict(case), "stream": _the_stream()}
    i = _inputs(case, seed, "cuda")
    torch.cuda.synchronize()   # the weights are built on the library's own streams
    if k == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        st.update(a=i["a"], w=_weight(i["w"], K, N), c=torch.empty(M, N, device="cuda"),
                  ws=_workspace(P.workspace_bytes(case["mode"], M, N, K)))
    elif k == "table":
        M, K, N = case["M"], case["K"], case["N"]
        st.update(i, c=torch.empty(M, N, device="cuda"), ws=_workspace(P.q8b_workspace_bytes(case["mode"], M, N, K)))
    elif k == "host":
        M, K, N = case["M"], case["K"], case["N"]
        w = {n: np.ascontiguousarray(i["w"][n].cpu().numpy()) for n in ("signs", "flags", "lo", "hi")}
        st.update(a=np.ascontiguousarray(i["a"].cpu().numpy()), w=w, c=np.empty((M, N), np.float32),
                  b=_FiveValueB(*(w[n].ctypes.data for n in ("signs", "flags", "lo", "hi")), None))
    elif k == "feed_forward":
        T, m = case["T"], case["mode"]
        st.update(x0=i["x"], x=torch.empty_like(i["x"]), gamma=i["gamma"], beta=i["beta"], l1=_weight(i["l1"], D, FF),
                  l2=_weight(i["l2"], FF, D), h=torch.empty(T, FF, device="cuda"),
                  q=P.DeviceBuffer(P.q_bytes(T, FF)), s=P.DeviceBuffer(4 * T),
                  ws=_workspace(max(P.q8a_workspace_bytes(m, T, FF, D), P.q8a_workspace_bytes(m, T, D, FF))))
    elif k == "attention":
        st.update(i, o=torch.empty(case["T"], D, device="cuda"))
    else:
        T, m = case["T"], case["mode"]
        blocks = [_dev_block(b) for b in i["blocks"]]
        st.update(x0=i["x"], x=i["x"].clone(), pe=i["pe"])
        if k == "block":
            st.update(block=blocks[0], ws=_workspace(P.block_workspace_bytes(m, T)))
        else:
            st.update(stack=P.Stack(blocks), ws=_workspace(P.stack_workspace_bytes(m, T, len(blocks))))
            torch.cuda.synchronize()
            with P.Graph(st["stream"]) as graph:
                st["stack"].run_dev(m, T, st["pe"].data_ptr(), st["x"].data_ptr(), st["ws"], st["stream"].ptr)
            st["graph"] = graph
    torch.cuda.synchronize()
    return st


class _FiveValueB(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("signs", "flags", "lo", "hi", "codes")]


_blas = None


def _drop_in():
    global _blas
    if _blas is None:
        _blas = C.CDLL(P.BLAS_SO)
        _blas.p2_sgemm_fvb.restype = None
        _blas.p2_sgemm_fvb.argtypes = [C.c_int, C.c_int, C.c_int, C.c_float, C.c_void_p, C.c_int, C.c_void_p, C.c_float,
                                       C.c_void_p, C.c_int]
    return _blas


def run(st):
    c, s = st["case"], st["stream"].ptr
    k = c["kind"]
    if k == "linear":
        P.fvb_gemm_dev(c["mode"], c["M"], c["N"], c["K"], 1.0, st["a"].data_ptr(), c["K"], st["w"], 0.0,
                       st["c"].data_ptr(), c["N"], st["ws"].ptr, st["ws"].nbytes, s)
        return st["c"]
    if k == "table":
        P.q8b_gemm_dev(c["mode"], c["M"], c["N"], c["K"], 1.0, st["a"].data_ptr(), c["K"], st["b"].data_ptr(), c["N"],
                       st["s"].data_ptr(), 0.0, st["c"].data_ptr(), c["N"], st["ws"].ptr, st["ws"].nbytes, s)
        return st["c"]
    if k == "host":
        _drop_in().p2_sgemm_fvb(c["M"], c["N"], c["K"], 1.0, st["a"].ctypes.data, c["K"], C.addressof(st["b"]), 0.0,
                                st["c"].ctypes.data, c["N"])
        return st["c"]
    if k == "attention":
        P._ok(P.hip().p2h_attention_rows(c["T"], st["qkv"].data_ptr(), st["bu"].data_ptr(), st["bv"].data_ptr(),
                                         st["p"].data_ptr(), st["o"].data_ptr(), s), "p2h_attention_rows")
        return st["o"]
    # the residual rows are updated in place: each pass starts on a fresh copy of them, as it would on a new window
    P._ok(P.hip().p2h_memcpy_d2d(st["x"].data_ptr(), st["x0"].data_ptr(), 4 * st["x"].numel(), s), "d2d")
    if k == "feed_forward":
        T, m, q, sc, ws = c["T"], c["mode"], st["q"].ptr, st["s"].ptr, st["ws"]
        P.layer_norm_quant_rows_dev(T, D, st["x"].data_ptr(), D, st["gamma"].data_ptr(), st["beta"].data_ptr(), q,
                                    P.q_ld(D), sc, s)
        P.fvb_gemm_q8a_silu_dev(m, T, FF, D, 1.0, q, P.q_ld(D), sc, st["l1"], st["h"].data_ptr(), ws.ptr, ws.nbytes, s)
        P.quant_rows_dev(T, FF, st["h"].data_ptr(), FF, q, P.q_ld(FF), sc, s)
        P.fvb_gemm_q8a_dev(m, T, D, FF, 0.5, q, P.q_ld(FF), sc, st["l2"], 1.0, st["x"].data_ptr(), D, ws.ptr, ws.nbytes,
                           s)
        return st["x"]
    if k == "block":
        st["block"].run_dev(c["mode"], c["T"], st["pe"].data_ptr(), st["x"].data_ptr(), st["ws"], s)
    else:
        st["graph"].launch()
    return st["x"]


# ── what a pass cannot do without ───────────────────────────────────────────────────────────────────────────────

def _linear_work(M, K, N, a=True, c=True):
    """Packed planes and lo, hi once; fp32 rows in and out where they are the pass's own."""
    return K * N * 3 // 8 + 8 * N + 4 * M * K * a + 4 * M * N * c, 2 * M * N * K


def _attention_flops(T):
    return H * DH * (2 * T * T + 2 * T * (2 * T - 1) + 2 * T * T)


def work(case):
    k = case["kind"]
    if k in ("linear", "host"):
        b, f = _linear_work(case["M"], case["K"], case["N"])
    elif k == "table":
        M, K, N = case["M"], case["K"], case["N"]
        b, f = K * N + 4 * N + 4 * M * K + 4 * M * N, 2 * M * N * K
    else:
        T = case["T"]
        if k == "feed_forward":
            parts = [_linear_work(T, D, FF, False, False), _linear_work(T, FF, D, False, False)]
            b, f = sum(p[0] for p in parts) + 8 * D + 8 * T * D, sum(p[1] for p in parts)
        elif k == "attention":
            b, f = 4 * T * 3 * D + 8 * D + 4 * (2 * T - 1) * D + 4 * T * D, _attention_flops(T)
        else:
            n = case.get("blocks", 1)
            parts = [_linear_work(2 * T - 1 if name == "pos" else T, K, N, False, False)
                     for name, (K, N) in P.BLOCK_LINEARS.items()]
            vec = 4 * (12 * D + D * P.CONV_K + D)
            b = n * (sum(p[0] for p in parts) + vec) + 8 * T * D + 4 * (2 * T - 1) * D
            f = n * (sum(p[1] for p in parts) + _attention_flops(T) + 2 * T * D * P.CONV_K)
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """fp32 sums of exact products everywhere; where rows are quantised between two steps of one pass (the
    feed-forward, the quantised block and window), a last-bit change of a row moves an int8 code now and then, and the
    steps after it carry the moved code on."""
    k, mode = case["kind"], case.get("mode")
    if mode == "exact":   # seen: linear 4.5e-7, table 1.1e-6 (a chain of K additions), 24 blocks 3e-7
        return {"rel": 5e-6 if k == "table" else 2e-6, "max": 5e-5}
    if k in ("linear", "table", "host"):   # seen: 6e-8 (whole-number sums, one rounding per 1024 rows)
        return {"rel": 5e-7, "max": 1e-5}
    if k == "attention":   # seen: 7e-7
        return {"rel": 3e-6, "max": 2e-4}
    if k == "feed_forward":   # seen: 5e-5, one code in a row of 4096 1.2e-2 of a value
        return {"rel": 2e-4, "max": 0.05}
    # seen: one block 1.1e-4, 24 blocks 5.4e-3 (and as much from one ulp on every input value)
    return {"rel": 1e-3, "max": 0.05} if k == "block" else {"rel": 0.02, "max": 0.4}


# ── the same in 64 bits ─────────────────────────────────────────────────────────────────────────────────────────

def _values(p, mode):
    """The weight as 64-bit values: {0, ±lo, ±hi}, or in the int8w mode its int8 codes (lo as the nearest 127th of hi)
    times hi / 127, which is that mode's format."""
    lo, hi = p["lo"].double(), p["hi"].double()
    if mode == "int8w":
        lo = torch.round(p["lo"] * 127.0 / p["hi"]).clamp(0, 127).double() * hi / 127.0
    return (p["code"].double() - 1.0) * torch.where(p["flag"] != 0, hi, lo)


def _quantised(a):
    """Rows as their int8 codes times the row's scale: the format both int8 modes multiply. The codes are found in the
    precision of the rows (32-bit rows: as the format's definition rounds them, the last K % 16 columns by the quotient
    itself). Quotients of two tensors: torch divides by a number through its reciprocal."""
    amax = a.abs().amax(1, keepdim=True)
    scale = amax / torch.full_like(amax, 127.0)
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    q = torch.round(a * (torch.ones_like(scale) / scale)).clamp(-128, 127)
    k16 = a.shape[1] // 16 * 16
    q[:, k16:] = torch.round(a[:, k16:] / scale).clamp(-127, 127)
    return q.double() * scale.double()


def _lin64(a, p, mode):
    return (a.double() if mode == "exact" else _quantised(a)) @ _values(p, mode)


def _ln64(x, g, b):
    m = x.mean(1, keepdim=True)
    v = ((x - m) ** 2).mean(1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * g.double() + b.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def _attention64(qkv, bu, bv, p):
    T = qkv.shape[0]
    q, k, v = (qkv[:, j * D:(j + 1) * D].double().view(T, H, DH).transpose(0, 1) for j in range(3))
    ph = p.double().view(2 * T - 1, H, DH).transpose(0, 1)
    ac = torch.matmul(q + bu.double().view(H, 1, DH), k.transpose(1, 2).contiguous())
    bd = torch.matmul(q + bv.double().view(H, 1, DH), ph.transpose(1, 2).contiguous())
    at = torch.arange(T, device=qkv.device)[None, :] + (T - 1) - torch.arange(T, device=qkv.device)[:, None]
    s = (ac + torch.gather(bd, 2, at.expand(H, T, T))) / math.sqrt(DH)
    return torch.matmul(torch.softmax(s, 2), v.contiguous()).transpose(0, 1).reshape(T, D)


def _feed_forward64(x, g, b, l1, l2, mode):
    return x + 0.5 * _lin64(_silu64(_lin64(_ln64(x, g, b), l1, mode)), l2, mode)


def _block64(x, pe, b, mode):
    T = x.shape[0]
    x = _feed_forward64(x, b["norm_ff1_w"], b["norm_ff1_b"], b["ff1_l1"], b["ff1_l2"], mode)
    qkv = _lin64(_ln64(x, b["norm_sa_w"], b["norm_sa_b"]), b["qkv"], mode)
    x = x + _lin64(_attention64(qkv, b["bias_u"], b["bias_v"], _lin64(pe, b["pos"], mode)), b["out"], mode)
    a, gate = _lin64(_ln64(x, b["norm_conv_w"], b["norm_conv_b"]), b["pw1"], mode).chunk(2, 1)
    padded = torch.nn.functional.pad(a * torch.sigmoid(gate), (0, 0, P.CONV_K // 2, P.CONV_K // 2))
    taps = b["dw_w"].double().view(D, P.CONV_K)
    conv = sum(padded[j:j + T] * taps[:, j] for j in range(P.CONV_K)) + b["dw_b"].double()
    x = x + _lin64(_silu64(conv), b["pw2"], mode)
    x = _feed_forward64(x, b["norm_ff2_w"], b["norm_ff2_b"], b["ff2_l1"], b["ff2_l2"], mode)
    return _ln64(x, b["norm_out_w"], b["norm_out_b"])


def exact(case, seed):
    k, mode = case["kind"], case.get("mode", "int8w")
    i = _inputs(case, seed, "cuda")
    if k in ("linear", "host"):
        out = _lin64(i["a"], i["w"], mode)
        return out.cpu().numpy() if k == "host" else out
    if k == "table":
        a = i["a"].double() if mode == "exact" else _quantised(i["a"])
        return a @ (i["b"].double() * i["s"].double())
    if k == "attention":
        return _attention64(i["qkv"], i["bu"], i["bv"], i["p"])
    if k == "feed_forward":
        return _feed_forward64(i["x"].double(), i["gamma"], i["beta"], i["l1"], i["l2"], mode)
    x = i["x"].double()
    for b in i["blocks"]:
        x = _block64(x, i["pe"], b, mode)
    return x
