"""What this framework's speed is measured on: the calls that an RWKV-7 serving engine makes, at its sizes.

Six kinds of pass, each through the package's public entry points:

    decode   one token for every running sequence: per layer timemix_prologue -> wkv7_pool_ -> timemix_epilogue, the
             layers captured once in a HIP graph and replayed for every token, as an engine's decode step is
    verify   a speculative step on one layer: StatePool.verify_ over T draft tokens with per-token snapshots, then
             StatePool.rollback_ to the accepted prefixes
    prefill  wkv7 on dense rows, from zero or given states, output and final states
    mixed    wkv7_pool_ on a packed batch of prefill rows and decode rows, in place in a slot pool
    timemix  timemix_prologue and timemix_epilogue over the tokens of a prefill
    linear   a layer's six quantised products (r, k, v, output, FFN up and down) with int6_matmul, on the bit planes or
             the packed layout, bf16 or fp16 activations; up to 256 rows the six are replayed from a HIP graph (a
             decode step's), above they are eager calls (a prefill's)

Head size 64.  H = 64 and F = 4 C (C = 4096) is the 7.2B shape, H = 40 the 2.9B one, H = 12 a 0.1B one, H = 8 one
rank's share of H = 64 on eight GPUs.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rwkv-infer-next_amd"))
from rwkv_next_amd import kernels  # noqa: E402

N = 64            # head size
GROUP_K = 128     # rows per scale of a quantised weight
GRAPH_MAX_M = 256  # up to here a linear pass is a decode step's and comes from a graph
EPS = 1e-5 * 64   # the model's group-norm epsilon


# ----------------------------------------------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one user chatting with a small model: latency and launches
        dict(name="decode_b1_h12", kind="decode", B=1, H=12, layers=12),
        # an odd number of running sequences on the 2.9B shape
        dict(name="decode_b23_h40", kind="decode", B=23, H=40, layers=8),
        # the serving batch on the 7.2B shape
        dict(name="decode_b64_h64", kind="decode", B=64, H=64, layers=4),
        # speculative decoding of the serving batch: verify five draft tokens, keep a prefix
        dict(name="verify_b64_t5_h64", kind="verify", B=64, T=5, H=64),
        # a short prompt on a small model
        dict(name="prefill_t500_h12", kind="prefill", B=1, T=500, H=12, state=False),
        # a long prompt on the 7.2B shape
        dict(name="prefill_t4096_h64", kind="prefill", B=1, T=4096, H=64, state=False),
        # a continuous-batching step: prompts of up to 2048 tokens beside running sequences
        dict(name="mixed_8x2048_d120_h64", kind="mixed", rows=8, max_len=2048, decode=120, H=64),
        # the elementwise work around the recurrence for a long prompt
        dict(name="timemix_t4096_h64", kind="timemix", T=4096, H=64),
        # one sequence's decode step on weights as the reference stores them
        dict(name="linear_m1_planes", kind="linear", M=1, C=4096, fmt="planes", dtype="bf16"),
        # the serving batch's decode step on packed weights
        dict(name="linear_m64_packed", kind="linear", M=64, C=4096, fmt="packed", dtype="bf16"),
        # a big batch of an odd size on the 2.9B shape, fp16 activations, weights as the reference stores them
        dict(name="linear_m203_planes_f16", kind="linear", M=203, C=2560, fmt="planes", dtype="f16"),
        # a prompt chunk through the quantised layers
        dict(name="linear_m2048_packed", kind="linear", M=2048, C=4096, fmt="packed", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "verify", "prefill", "prefill", "mixed", "timemix", "linear", "linear",
                       "linear"))
    H = rng.choice((8, 12, 40, 64))
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 64), H=H, layers=rng.randint(2, 4) if H == 64 else rng.randint(4, 12))
    if kind == "verify":
        return dict(kind=kind, B=_log_int(rng, 1, 64), T=rng.randint(2, 8) if H < 64 else rng.randint(2, 5), H=H)
    if kind == "prefill":
        T = _log_int(rng, 33, 4096)
        return dict(kind=kind, B=rng.randint(1, max(1, min(8, 4096 // T))), T=T, H=H, state=rng.random() < 0.5)
    if kind == "mixed":
        return dict(kind=kind, rows=rng.randint(1, 8), max_len=_log_int(rng, 40, 2048), decode=rng.randint(0, 120), H=H)
    if kind == "timemix":
        return dict(kind=kind, T=_log_int(rng, 1, 4096), H=H)
    return dict(kind=kind, M=_log_int(rng, 1, 2048), C=N * rng.choice((12, 40, 64)),
                fmt=rng.choice(("planes", "packed")), dtype=rng.choice(("bf16", "bf16", "f16")))


# ----------------------------------------------------------------------------------------------------------------
# inputs, made from the seed on the GPU
# ----------------------------------------------------------------------------------------------------------------
class _Draws:
    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(int(seed))
        self.cpu = torch.Generator().manual_seed(int(seed))  # lengths and slots, which a scheduler has on the host

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, device=self.dev, generator=self.g) * std + mean

    def bf16(self, *shape, std=1.0, mean=0.0):
        return self.normal(*shape, std=std, mean=mean).to(torch.bfloat16)

    def perm(self, n):
        return torch.randperm(n, generator=self.cpu).to(self.dev)


def _operands(x, B, T, H):
    """The six operands of the recurrence with the model's value ranges: r, k, v ~ N(0, 1), raw w in (-inf, -0.5),
    a = -kappa, b = kappa * gate with kappa of unit length per head."""
    C = H * N
    r, k, v = (x.bf16(B, T, C) for _ in range(3))
    w = (-torch.nn.functional.softplus(x.normal(B, T, C, std=2.0)) - 0.5).to(torch.bfloat16)
    kap = torch.nn.functional.normalize(x.normal(B, T, H, N), dim=-1).view(B, T, C)
    return [r, w, k, v, (-kap).to(torch.bfloat16), (kap * torch.sigmoid(x.normal(B, T, C))).to(torch.bfloat16)]


def _layer(x, M, H):
    """One layer's projections and per-channel parameters."""
    C = H * N
    return dict(r=x.bf16(M, C), k=x.bf16(M, C), v=x.bf16(M, C), o=x.bf16(3, M, C, std=0.5), v_first=x.bf16(M, C),
                g=x.bf16(M, C, std=0.5), b_w=x.bf16(1, C, std=0.5), b_a=x.bf16(1, C, std=0.5),
                b_v=x.bf16(1, C, std=0.5), kk_mul=x.bf16(1, C, std=0.5, mean=1.0), ka_mul=x.bf16(1, C, std=0.3),
                lnx_w=x.bf16(C, std=0.2, mean=1.0), lnx_b=x.bf16(C, std=0.1), r_k=x.bf16(H, N, std=0.3))


def _mixed_lens(case):
    """Row lengths: prefill rows of 2..max_len tokens among decode rows, the same for every seed."""
    g = torch.Generator().manual_seed(case["rows"] + 100 * case["decode"] + 100000 * case["max_len"])
    lens = torch.randint(2, case["max_len"] + 1, (case["rows"],), generator=g).tolist() + [1] * case["decode"]
    return [lens[i] for i in torch.randperm(len(lens), generator=g).tolist()]


def _mixed_rows(x, case):
    """Row lengths, their prefix sums, which rows start fresh (every second prefill row) and the slots."""
    lens = _mixed_lens(case)
    n, cu = len(lens), [0]
    for t in lens:
        cu.append(cu[-1] + t)
    fresh = [t > 1 and i % 2 == 0 for i, t in enumerate(lens)]
    return lens, torch.tensor(cu, dtype=torch.int32, device=x.dev), torch.tensor(fresh, device=x.dev), x.perm(2 * n)[:n]


def _products(case):
    """(K, N) of the layer's six products."""
    C, F = case["C"], 4 * case["C"]
    return [(C, C)] * 4 + [(C, F), (F, C)]


def _codes(x, K, n):
    """6-bit codes u = q + 32 (K, n) of normal weights quantised by their group's largest magnitude, and fp16 scales."""
    u = (x.normal(K, n, std=11.5).round_().clamp_(-32, 31) + 32).to(torch.uint8)
    s = (torch.exp(x.normal(K // GROUP_K, n, std=0.2)) / (11.5 * math.sqrt(K))).half()
    return u, s


def _pack_planes(u):
    """The bit planes of the weight format: per 64-row chunk, 32 rows of low nibbles and 16 rows of top bits."""
    K, n = u.shape
    c = u.view(K // 64, 64, n)
    lo = (c[:, :32] & 15) | ((c[:, 32:] & 15) << 4)
    h = c >> 4
    hi = h[:, :16] | (h[:, 16:32] << 2) | (h[:, 32:48] << 4) | (h[:, 48:] << 6)
    return lo.reshape(K // 2, n).contiguous(), hi.reshape(K // 4, n).contiguous()


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def _activations(x, case):
    """Inputs of the six products: C features each, the last 4 C."""
    return [x.normal(case["M"], k).to(_dtype(case)) for k, _ in _products(case)]


def _inputs(case, seed):
    x = _Draws(seed)
    kind, d = case["kind"], {}
    if kind == "decode":
        B, H, L = case["B"], case["H"], case["layers"]
        d["layers"] = [_layer(x, B, H) for _ in range(L)]
        d["slots"] = x.perm(2 * B)[:B]
        d["pool"] = x.normal(L, 2 * B, H, N, N, std=0.1)
    elif kind == "verify":
        B, T, H = case["B"], case["T"], case["H"]
        d["ops"] = _operands(x, B, T, H)
        d["slots"] = x.perm(2 * B)[:B]
        d["pool"] = x.normal(1, 2 * B, H, N, N, std=0.1)
        d["n"] = torch.randint(1, T + 1, (B,), generator=x.cpu).to(x.dev)
    elif kind == "prefill":
        d["ops"] = _operands(x, case["B"], case["T"], case["H"])
        d["h0"] = x.normal(case["B"], case["H"], N, N, std=0.1) if case["state"] else None
    elif kind == "mixed":
        d["lens"], d["cu"], d["fresh"], d["slots"] = _mixed_rows(x, case)
        d["ops"] = _operands(x, 1, sum(d["lens"]), case["H"])
        d["pool"] = x.normal(2 * len(d["lens"]), case["H"], N, N, std=0.1)
    elif kind == "timemix":
        d = _layer(x, case["T"], case["H"])
        d["y"] = x.bf16(case["T"], case["H"] * N)
    else:
        d["codes"] = [_codes(x, k, n) for k, n in _products(case)]
        d["a"] = _activations(x, case)
    return d


# ----------------------------------------------------------------------------------------------------------------
# the passes
# ----------------------------------------------------------------------------------------------------------------
def _decode_step(s):
    """Every layer's time-mix for one token of each sequence; returns the layers' inputs of the output projection."""
    H, out = s["H"], []
    for i, p in enumerate(s["layers"]):
        B, C = p["r"].shape
        ins, _ = kernels.timemix_prologue(p["r"], p["k"], p["v"], p["o"], p["v_first"], p["b_w"], p["b_a"], p["b_v"],
                                          p["kk_mul"], p["ka_mul"], H, N, i == 0)
        y = kernels.wkv7_pool_(*[t.view(B, 1, C) for t in ins], s["pool"].layer(i), s["slots"], H, N)
        out.append(kernels.timemix_epilogue(y.view(B, C), p["r"], ins[2], ins[3], p["g"], p["lnx_w"], p["lnx_b"],
                                            p["r_k"], H, N, EPS))
    return out


def _products_step(s):
    return [kernels.int6_matmul(a, *w) for a, w in zip(s["a"], s["weights"])]


def _captured(step, s):
    """The step captured in a HIP graph after one eager warm-up, and its outputs (written by every replay)."""
    step(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(s)
    return graph, out


def prepare(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    s = dict(kind=kind, H=case.get("H"))
    if kind == "decode":
        s.update(layers=d["layers"], slots=d["slots"],
                 pool=kernels.StatePool(case["layers"], 2 * case["B"], case["H"], "cuda"))
        s["graph"], s["out"] = _captured(_decode_step, s)
        s["pool"].wkv.copy_(d["pool"])  # after the warm-up, which updated its zero states
    elif kind == "verify":
        s.update(ops=d["ops"], slots=d["slots"], n=d["n"],
                 pool=kernels.StatePool(1, 2 * case["B"], case["H"], "cuda"))
        s["pool"].wkv.copy_(d["pool"])
        s["snapshots"] = s["pool"].snapshot_buffer(case["B"], case["T"])
    elif kind == "mixed":
        s.update(d, max_len=case["max_len"])
    elif kind == "linear":
        s["a"] = d["a"]
        planes = [(*_pack_planes(u), sc, GROUP_K) for u, sc in d["codes"]]
        s["weights"] = planes if case["fmt"] == "planes" else [(kernels.prepack_int6(*p),) for p in planes]
        if case["M"] <= GRAPH_MAX_M:
            s["graph"], s["out"] = _captured(_products_step, s)
    else:
        s.update(d)
    return s


def run(s):
    kind, H = s["kind"], s["H"]
    if kind == "decode":
        s["graph"].replay()
        return s["out"], s["pool"].wkv
    if kind == "verify":
        o = s["pool"].verify_(0, *s["ops"], s["slots"], s["snapshots"])
        s["pool"].rollback_(s["slots"], s["n"], s["snapshots"])
        return o, s["snapshots"], s["pool"].wkv
    if kind == "prefill":
        return kernels.wkv7(*s["ops"], s["h0"], H, N)
    if kind == "mixed":
        o = kernels.wkv7_pool_(*s["ops"], s["pool"], s["slots"], H, N, cu_seqlens=s["cu"], fresh=s["fresh"],
                               max_len=s["max_len"])
        return o, s["pool"]
    if kind == "timemix":
        ins, _ = kernels.timemix_prologue(s["r"], s["k"], s["v"], s["o"], s["v_first"], s["b_w"], s["b_a"], s["b_v"],
                                          s["kk_mul"], s["ka_mul"], H, N, False)
        out = kernels.timemix_epilogue(s["y"], s["r"], ins[2], ins[3], s["g"], s["lnx_w"], s["lnx_b"], s["r_k"], H, N,
                                       EPS)
        return list(ins[1:]), out
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    return _products_step(s)


# ----------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------------------------
STATE = N * N * 4      # bytes of one state
STEP_FLOPS = 9 * N * N  # of one token of one head: decay, a^T S, the two outer products, S^T r
PROLOGUE, EPILOGUE = 22, 12  # bytes per (token, channel): 6 read + 5 written; 5 read + 1 written, bf16


def work(case):
    kind, H = case["kind"], case.get("H", 0)
    if kind == "decode":
        # the six operands are made and used inside the pass: only the projections, the states and the results count
        n = case["B"] * case["layers"] * H
        return dict(bytes=n * (2 * STATE + N * 2 * 9), flops=n * (STEP_FLOPS + 60 * N))
    if kind == "verify":
        B, T = case["B"], case["T"]
        return dict(bytes=B * H * (STATE + T * (STATE + N * 14) + 2 * STATE), flops=B * H * T * STEP_FLOPS)
    if kind == "prefill":
        rows, tokens = case["B"], case["B"] * case["T"]
        return dict(bytes=H * (tokens * N * 14 + rows * STATE * (2 if case["state"] else 1)),
                    flops=H * tokens * STEP_FLOPS)
    if kind == "mixed":
        n = case["rows"] + case["decode"]
        tokens = sum(_mixed_lens(case))
        return dict(bytes=H * (tokens * N * 14 + n * 2 * STATE), flops=H * tokens * STEP_FLOPS)
    if kind == "timemix":
        n = case["T"] * H * N
        return dict(bytes=n * (PROLOGUE + EPILOGUE - 4), flops=60 * n)  # k' and v' are written and read within the pass
    M = case["M"]
    return dict(bytes=sum(k * n * 3 / 4 + k // GROUP_K * n * 2 + 2 * M * (k + n) for k, n in _products(case)),
                flops=sum(2 * M * k * n for k, n in _products(case)))


# About four times what the passes are off the 64-bit values.  A value rounded once to bf16 is 1.7e-3 off (2-norm;
# largest 2^-8), to fp16 an eighth of that; the chunked recurrence multiplies bf16 operands for its outputs (3.7e-3,
# largest 0.035), and above 256 rows the weight itself is rounded to the activations' type (2.4e-3, largest 0.012).
def tolerance(case):
    kind = case["kind"]
    if kind in ("prefill", "mixed"):
        return dict(rel=1.5e-2, max=0.14)
    if kind in ("decode", "timemix"):  # the largest differences: group norms of values that nearly cancel
        return dict(rel=7e-3, max=0.06)
    if kind == "verify":
        return dict(rel=7e-3, max=0.02)
    unit = 1.0 if case["dtype"] == "bf16" else 0.125
    return dict(rel=1e-2 * unit, max=0.05 * unit) if case["M"] > GRAPH_MAX_M else dict(rel=7e-3 * unit, max=0.02 * unit)


# ----------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ----------------------------------------------------------------------------------------------------------------
def _prologue64(p, H, first):
    f = {n: t.double() for n, t in p.items()}
    M = f["k"].shape[0]
    w = -torch.nn.functional.softplus(-(f["b_w"] + f["o"][1])) - 0.5
    a = torch.sigmoid(f["b_a"] + f["o"][2])
    v = f["v"] if first else f["v"] + (f["v_first"] - f["v"]) * torch.sigmoid(f["b_v"] + f["o"][0])
    kk = torch.nn.functional.normalize((f["k"] * f["kk_mul"]).view(M, H, N), dim=-1).view(M, H * N)
    return [f["r"], w, f["k"] * (1 + (a - 1) * f["ka_mul"]), v, -kk, kk * a]


def _epilogue64(y, r, k, v, p, H):
    M = y.shape[0]
    x = torch.nn.functional.group_norm(y, H, p["lnx_w"].double(), p["lnx_b"].double(), EPS)
    bonus = (r.view(M, H, N) * k.view(M, H, N) * p["r_k"].double()).sum(-1, keepdim=True)
    return (x + (bonus * v.view(M, H, N)).view(M, H * N)) * p["g"].double()


def _recurrence64(ops, S, H, lens=None, each=None):
    """(o (B, T, H*N), final states) from S (B, H, N, N), over the first lens[b] tokens of row b; `each(t, S)` is
    called with the states after every token."""
    B, T = ops[0].shape[:2]
    r, w, k, v, a, b = (t.double().view(B, T, H, N) for t in ops)
    d = torch.exp(-torch.exp(w))
    o = torch.zeros(B, T, H, N, dtype=torch.float64, device=S.device)
    n = B
    for t in range(T):
        if lens is not None:  # rows come longest first: the ones that go on are the first n
            while lens[n - 1] <= t:
                n -= 1
        Q = S[:n]
        sa = torch.matmul(a[:n, t, :, None, :], Q)
        Q = Q * d[:n, t, :, :, None] + b[:n, t, :, :, None] * sa + k[:n, t, :, :, None] * v[:n, t, :, None, :]
        o[:n, t] = torch.matmul(r[:n, t, :, None, :], Q)[:, :, 0]
        if n < B:
            S[:n] = Q
        else:
            S = Q
        if each is not None:
            each(t, S)
    return o.view(B, T, H * N), S


def exact(case, seed):
    d, kind, H = _inputs(case, seed), case["kind"], case.get("H")
    rounded = lambda t: t.to(torch.bfloat16).double()  # what one entry point hands to the next is bf16
    if kind == "decode":
        pool, out = d["pool"].double(), []
        for i, p in enumerate(d["layers"]):
            B, C = p["r"].shape
            ins = [rounded(t) for t in _prologue64(p, H, i == 0)]
            y, S = _recurrence64([t.view(B, 1, C) for t in ins], pool[i][d["slots"]], H)
            pool[i][d["slots"]] = S
            out.append(_epilogue64(rounded(y).view(B, C), ins[0], ins[2], ins[3], p, H))
        return out, pool
    if kind == "verify":
        pool = d["pool"].double()
        snaps = torch.empty(1, case["B"], case["T"], H, N, N, dtype=torch.float64, device=pool.device)

        def keep(t, S):
            snaps[0, :, t] = S
        o, _ = _recurrence64(d["ops"], pool[0][d["slots"]], H, each=keep)
        pool[0][d["slots"]] = snaps[0, torch.arange(case["B"], device=pool.device), d["n"] - 1]
        return o, snaps, pool
    if kind == "prefill":
        h0 = d["h0"].double() if case["state"] else d["ops"][0].new_zeros(case["B"], H, N, N, dtype=torch.float64)
        return _recurrence64(d["ops"], h0, H)
    if kind == "mixed":
        lens, T, cu = d["lens"], max(d["lens"]), d["cu"].tolist()
        order = sorted(range(len(lens)), key=lambda i: -lens[i])
        ops = []
        for x in d["ops"]:  # rows padded to the longest, longest first
            pad = x.new_zeros(len(lens), T, H * N)
            for j, i in enumerate(order):
                pad[j, :lens[i]] = x[0, cu[i]:cu[i + 1]]
            ops.append(pad)
        rows = torch.tensor(order, device=d["slots"].device)
        pool = d["pool"].double()
        S = pool[d["slots"][rows]]
        S[d["fresh"][rows]] = 0
        y, S = _recurrence64(ops, S, H, lens=[lens[i] for i in order])
        pool[d["slots"][rows]] = S
        o = y.new_empty(1, cu[-1], H * N)
        for j, i in enumerate(order):
            o[0, cu[i]:cu[i + 1]] = y[j, :lens[i]]
        return o, pool
    if kind == "timemix":
        ins = _prologue64(d, H, False)
        return ins[1:], _epilogue64(d["y"].double(), ins[0], rounded(ins[2]), rounded(ins[3]), d, H)
    out = []
    for a, (u, sc) in zip(d["a"], d["codes"]):
        q = (u.double() - 32).view(sc.shape[0], GROUP_K, -1) * sc.double()[:, None]
        out.append(torch.matmul(a.double(), q.view(u.shape[0], -1)))
    return out
