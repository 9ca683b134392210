"""Timed cases of the W4A16 MoE expert path, through its public entry points.

Shapes are the ones this repository's benchmark and tests use (hidden / expert
width / group: 2048/512/128, 2560/640/64, 3072/768/64, 512 experts, top-10; the
2048 -> 4096 W4A16 and 2048 -> 8192 W8A16 projections), over the token counts a
serving program meets: one token, a few sequences decoding together, a short
prompt, a prompt chunk, and a long prefill. Calls of up to a few dozen rows are
what such a program captures in a HIP graph over its layers (each layer with
weights of its own), so those cases replay one; the others call eagerly.

Inputs are made on the device from the seed: int4 nibbles and int8 weights
uniform, scales bf16(|N(0,1)| * 0.02) (W8: * 0.004), activations and router
logits bf16(N(0,1)), skewed routing as Zipf popularity plus Gumbel noise.
"""
import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "qwen-ascend_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF16 = torch.bfloat16

# (hidden, expert width, scale group) of the configurations in bench.py
SHAPES = ((2048, 512, 128), (2560, 640, 64), (3072, 768, 64))


def listed():
    return [
        # one sequence decoding: the expert block of 8 layers in one captured
        # step, weights also laid out as decode tiles at load time
        {"name": "decode_b1_8layers", "kind": "experts", "T": 1, "H": 2048, "MI": 512, "gs": 128, "E": 512, "k": 10,
         "zipf": 0.0, "shared": False, "tiles": True, "layers": 8, "graph": True},
        # four sequences decoding together with the gated shared-expert merge,
        # straight from the int4pack container
        {"name": "decode_b4_4layers", "kind": "experts", "T": 4, "H": 2560, "MI": 640, "gs": 64, "E": 512, "k": 10,
         "zipf": 0.0, "shared": True, "tiles": False, "layers": 4, "graph": True},
        # a short prompt (or a batch of decoding sequences): most experts that
        # are read serve a single row
        {"name": "prompt_t23", "kind": "experts", "T": 23, "H": 2560, "MI": 640, "gs": 64, "E": 512, "k": 10,
         "zipf": 0.0, "shared": True, "tiles": False, "layers": 1, "graph": False},
        # a prompt chunk with skewed expert popularity
        {"name": "prefill_t512_zipf", "kind": "experts", "T": 512, "H": 2048, "MI": 512, "gs": 128, "E": 512, "k": 10,
         "zipf": 1.1, "shared": False, "tiles": False, "layers": 1, "graph": False},
        # a long prefill at the widest configuration: the largest case
        {"name": "prefill_t4096", "kind": "experts", "T": 4096, "H": 3072, "MI": 768, "gs": 64, "E": 512, "k": 10,
         "zipf": 0.0, "shared": True, "tiles": False, "layers": 1, "graph": False},
        # one projection of one token, called eagerly: the smallest call
        {"name": "w4_proj_m1", "kind": "w4", "M": 1, "K": 2048, "N": 4096, "gs": 128, "layers": 1, "graph": False},
        # the same projection for a batch of decoding sequences, over 8 layers
        {"name": "w4_proj_m48_8layers", "kind": "w4", "M": 48, "K": 2048, "N": 4096, "gs": 128, "layers": 8,
         "graph": True},
        # a dense int8 projection for a few sequences (ragged row count) ...
        {"name": "w8_dense_m7_8layers", "kind": "w8", "M": 7, "K": 2048, "N": 8192, "gs": 128, "layers": 8,
         "graph": True},
        # ... and for a prompt chunk
        {"name": "w8_dense_m512", "kind": "w8", "M": 512, "K": 2048, "N": 8192, "gs": 128, "layers": 1,
         "graph": False},
        # shared expert and router projections of a short prompt chunk
        {"name": "shared_router_t200", "kind": "shared", "T": 200, "H": 2560, "MI": 640, "E": 512, "layers": 1,
         "graph": False},
        # the ordered weighted combine of a full prefill chunk
        {"name": "combine_t8192", "kind": "combine", "T": 8192, "k": 10, "H": 2560},
        # load time: one layer's experts from the LQP artifact to int4pack
        {"name": "convert_layer", "kind": "convert", "H": 2560, "MI": 640, "gs": 64, "E": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_mult(rng, lo, hi, step):
    return max(lo, min(hi, _log_int(rng, lo, hi) // step * step))


def draw(rng):
    kind = rng.choice(["experts", "experts", "experts", "experts", "w4", "w8", "w8", "shared", "combine", "convert"])
    if kind == "experts":
        if rng.random() < 0.5:
            H, MI, gs = rng.choice(SHAPES)
            E, k = 512, 10
        else:  # widths, expert counts and groups the tests use beside those
            gs = rng.choice([32, 64, 128])
            H, MI = _log_mult(rng, 512, 3072, 128), _log_mult(rng, 256, 768, 128)
            E, k = rng.choice([64, 128, 256, 512]), rng.choice([6, 8, 10])
        T = _log_int(rng, 1, 4096)
        small = T <= 48
        return {"kind": kind, "T": T, "H": H, "MI": MI, "gs": gs, "E": E, "k": k,
                "zipf": rng.choice([0.0, 0.0, round(rng.uniform(0.6, 1.2), 2)]), "shared": rng.random() < 0.5,
                "tiles": T <= 4 and rng.random() < 0.5, "layers": rng.choice([2, 3, 4]) if small else 1,
                "graph": small}
    if kind in ("w4", "w8"):
        gs = rng.choice([32, 64, 128])
        M = _log_int(rng, 1, 2048 if kind == "w8" else 512)
        small = M <= 64 and rng.random() < 0.8
        return {"kind": kind, "M": M, "K": _log_mult(rng, 512, 4096, 128),
                "N": _log_mult(rng, 512, 8192, 32 if kind == "w4" else 16), "gs": gs,
                "layers": rng.choice([4, 6, 8]) if small else 1, "graph": small}
    if kind == "shared":
        H, MI, _ = rng.choice(SHAPES)
        T = _log_int(rng, 1, 4096)
        return {"kind": kind, "T": T, "H": H, "MI": MI, "E": rng.choice([64, 256, 512]),
                "layers": 4 if T <= 48 else 1, "graph": T <= 48}
    if kind == "combine":
        return {"kind": kind, "T": _log_int(rng, 64, 8192), "k": rng.choice([6, 8, 10]),
                "H": rng.choice([2048, 2560, 3072])}
    H, MI, gs = rng.choice(SHAPES)
    return {"kind": kind, "H": H, "MI": MI, "gs": gs, "E": rng.choice([64, 96, 128, 256, 320, 384])}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _words(g, shape):
    n = math.prod(shape)
    return torch.empty(4 * n, dtype=torch.uint8, device="cuda").random_(0, 256, generator=g).view(torch.int32).view(shape)


def _normal(g, shape, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(BF16)


def _scales(g, shape, std=0.02):
    return (torch.randn(shape, generator=g, device="cuda").abs_() * std).to(BF16)


def _logits(g, T, E, zipf):
    if not zipf:
        return _normal(g, (T, E))
    rank = torch.empty(E, device="cuda", dtype=torch.float64)
    rank[torch.randperm(E, generator=g, device="cuda")] = torch.arange(1, E + 1, device="cuda", dtype=torch.float64)
    logp = (-zipf * rank.log()).log_softmax(0)
    u = torch.rand((T, E), generator=g, device="cuda", dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    return (logp[None, :] - (-u.log()).log()).to(BF16)


def _data(case, seed):
    """The tensors of a case, made from the seed alone: one tuple per layer."""
    g, kind = _gen(seed), case["kind"]
    out = []
    for _ in range(case.get("layers", 1)):
        if kind == "experts":
            T, H, MI, gs, E = (case[v] for v in ("T", "H", "MI", "gs", "E"))
            shared = gate = None
            if case["shared"]:
                shared = _normal(g, (T, H), 0.5)
                gate = _normal(g, (T, 1)) if T <= 4 else None
            out.append((_words(g, (E, H, 2 * MI // 8)), _scales(g, (E, H // gs, 2 * MI)), _words(g, (E, MI, H // 8)),
                        _scales(g, (E, MI // gs, H)), _normal(g, (T, H)), _logits(g, T, E, case["zipf"]), shared, gate))
        elif kind == "w4":
            M, K, N, gs = (case[v] for v in ("M", "K", "N", "gs"))
            out.append((_normal(g, (M, K)), _words(g, (K, N // 8)), _scales(g, (K // gs, N))))
        elif kind == "w8":
            M, K, N, gs = (case[v] for v in ("M", "K", "N", "gs"))
            out.append((_normal(g, (M, K)), _words(g, (N, K // 4)).view(torch.int8), _scales(g, (N, K // gs), 0.004)))
        elif kind == "shared":
            T, H, MI, E = (case[v] for v in ("T", "H", "MI", "E"))
            out.append((_normal(g, (T, H)), _normal(g, (2 * MI + 1 + E, H), 0.02), _normal(g, (H, MI), 0.02)))
        elif kind == "combine":
            T, k, H = case["T"], case["k"], case["H"]
            out.append((_normal(g, (T * k, H)), torch.rand((T, k), generator=g, device="cuda").to(BF16),
                        torch.randperm(T * k, generator=g, device="cuda")))
        else:  # convert: the LQP tensors of both projections
            H, MI, gs, E = (case[v] for v in ("H", "MI", "gs", "E"))
            for N, K in ((2 * MI, H), (H, MI)):
                out.append((_words(g, (E, N, K // 8)).view(torch.uint8).view(E, N, K // 2),
                            torch.randint(1, 128, (E, N, K // gs), generator=g, device="cuda", dtype=torch.int8),
                            (torch.rand((E, N), generator=g, device="cuda") * 2e-4 + 1e-5).to(torch.float16)))
    return out


def prepare(case, seed):
    data, kind = _data(case, seed), case["kind"]
    if kind == "experts":
        from qmoe import ExpW4, moe_experts
        calls = []
        for gw, gsc, dw, dsc, x, lg, sh, gate in data:
            gu, dn = ExpW4.from_scales(gw, gsc), ExpW4.from_scales(dw, dsc)
            if case["tiles"]:
                gu.decode_tiles("gate_up")
                dn.decode_tiles("down")
            calls.append(lambda x=x, lg=lg, gu=gu, dn=dn, sh=sh, gate=gate: moe_experts(
                x, lg, gu, dn, case["k"], shared=sh, shared_gate=gate))
    elif kind == "w4":
        from qmoe import weight_quant_batchmatmul
        calls = [lambda x=x, w=w, s=s: weight_quant_batchmatmul(x, w, s, antiquant_group_size=case["gs"])
                 for x, w, s in data]
    elif kind == "w8":
        from qmoe import DenseW8
        calls = [lambda x=x, m=DenseW8(q, s): m(x) for x, q, s in data]
    elif kind == "shared":
        from qmoe.shared import gate_shared, shared_router

        def block(x, w, d):
            sh, gate2, logits = shared_router(x, w, d, case["MI"])
            if case["T"] <= 4:  # the decode block merges and gates inside the expert launch
                return sh, gate2, logits
            return sh, gate2, logits, gate_shared(sh, gate2)
        calls = [lambda x=x, w=w, d=d: block(x, w, d) for x, w, d in data]
    elif kind == "combine":
        from qmoe import weighted_reduce
        calls = [lambda x=x, w=w, inv=inv: weighted_reduce.reduce(x, w, inverse=inv) for x, w, inv in data]
    else:
        from qmoe.artifact import exp_w4_from_lqp

        def convert(v, s, b):
            e = exp_w4_from_lqp(v, s, b)
            return e.w4, e._scales
        calls = [lambda v=v, s=s, b=b: convert(v, s, b) for v, s, b in data]
    state = {"calls": calls}
    if case.get("graph"):
        for c in calls:  # eager first, as every program that captures does
            c()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = [c() for c in calls]
        state["graph"] = graph
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return [c() for c in state["calls"]]


# ---------------------------------------------------------------- what a pass cannot do without

def _distinct(E, k, T, zipf):
    """Expected number of experts that T tokens' top-k choices reach: each
    expert is in a token's choice with probability 1 - exp(-c p_e), c such that
    these sum to k."""
    p = [r ** -zipf for r in range(1, E + 1)]
    s = sum(p)
    p = [v / s for v in p]
    lo, hi = 0.0, 1e9
    for _ in range(200):
        c = (lo + hi) / 2
        if sum(1 - math.exp(-c * v) for v in p) < k:
            lo = c
        else:
            hi = c
    return sum(1 - math.exp(-c * v * T) for v in p)


def work(case):
    kind, L = case["kind"], case.get("layers", 1)
    if kind == "experts":
        T, H, MI, gs, E, k = (case[v] for v in ("T", "H", "MI", "gs", "E", "k"))
        per = (H * 2 * MI + MI * H) // 2 + (H // gs * 2 * MI + MI // gs * H) * 2
        b = _distinct(E, k, T, case["zipf"]) * per + T * (2 * H + E + (H if case["shared"] else 0)) * 2
        return {"bytes": L * b, "flops": L * 2.0 * T * k * 3 * H * MI}
    if kind in ("w4", "w8"):
        M, K, N, gs = (case[v] for v in ("M", "K", "N", "gs"))
        return {"bytes": L * (K * N // (2 if kind == "w4" else 1) + K // gs * N * 2 + M * (K + N) * 2.0),
                "flops": L * 2.0 * M * K * N}
    if kind == "shared":
        T, H, MI, E = (case[v] for v in ("T", "H", "MI", "E"))
        n1 = 2 * MI + 1 + E
        return {"bytes": L * 2.0 * (n1 * H + H * MI + T * (H + 1 + E + (1 if T <= 4 else 2) * H)),
                "flops": L * 2.0 * T * (n1 * H + H * MI)}
    if kind == "combine":
        T, k, H = case["T"], case["k"], case["H"]
        return {"bytes": T * k * H * 2 + T * k * 10 + T * H * 2.0, "flops": 2.0 * T * k * H}
    H, MI, gs, E = (case[v] for v in ("H", "MI", "gs", "E"))
    # int4 in and out; int8 scales and fp16 base in, the bf16 scales out
    return {"bytes": E * (3 * H * MI // 2 * 2 + 3 * H * MI // gs * 3 + (2 * MI + H) * 2.0), "flops": 0.0}


# Largest relative error of another correct implementation: bf16 results whose
# fp32 sums run in another order differ where a sum falls on the other side of
# a rounding boundary (one bf16 step, at most 2^-7 of the value). Through the
# expert block such a step travels on from gate/up, act and down. Measured
# against sums in 64 bits with the same bf16 rounding points: up to 4e-5 for
# the projections (more where a call has few outputs and one of them steps),
# 1.5e-4 for the shared expert, 2e-5 to 9e-4 for the expert blocks.
def tolerance(case):
    kind = case["kind"]
    if kind in ("combine", "convert"):  # fixed order of the sum, whole numbers: the same bits
        return "exact"
    if kind in ("w4", "w8"):
        return {"rel": 1e-3, "max": 0.01}
    return {"rel": 4e-3 if kind == "experts" else 1e-3}


# ---------------------------------------------------------------- the same in 64 bits

def _r(v):
    """bf16 rounding of a 64-bit value, as the operation prescribes at this point."""
    return v.to(BF16).double()


def _unpack4(w):
    """int4pack words [..., N/8] -> float64 [..., N]."""
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = (w.unsqueeze(-1) >> sh) & 15
    return ((q ^ 8) - 8).flatten(-2).double()


def _deq4(w, s):
    K, G = w.shape[0], s.shape[0]
    return (_unpack4(w).view(G, K // G, -1) * s.double().unsqueeze(1)).view(K, -1)


def _exact_experts(case, layer):
    gw, gsc, dw, dsc, x, lg, shared, gate = layer
    T, H, MI, k = case["T"], case["H"], case["MI"], case["k"]
    # equal logits go to the lower expert id
    idx = torch.sort(lg.float(), dim=1, descending=True, stable=True)[1][:, :k]
    p = lg.double().softmax(1).gather(1, idx)
    wt = _r(p / p.sum(1, keepdim=True))
    xd = x.double()
    prod = torch.zeros((T * k, H), dtype=torch.float64, device=x.device)
    flat = idx.reshape(-1)
    order = torch.sort(flat, stable=True)[1]
    counts = torch.bincount(flat, minlength=case["E"]).tolist()
    at = 0
    for e, n in enumerate(counts):
        if not n:
            continue
        rows = order[at:at + n]
        at += n
        gu = _r(xd[rows // k] @ _deq4(gw[e], gsc[e]))
        g, u = gu[:, :MI], gu[:, MI:]
        y = _r(_r(g / (1 + (-g).exp()) * u) @ _deq4(dw[e], dsc[e]))
        prod[rows] = _r(y * wt.reshape(-1)[rows].unsqueeze(1))
    out = prod.view(T, k, H).sum(1)
    if shared is None:
        return out
    sh = shared.double()
    if gate is not None:
        sh = _r(sh * _r(gate.double().sigmoid()))
    return _r(out) + sh


def exact(case, seed):
    kind, out = case["kind"], []
    for layer in _data(case, seed):
        if kind == "experts":
            out.append(_exact_experts(case, layer))
        elif kind == "w4":
            x, w, s = layer
            out.append(x.double() @ _deq4(w, s))
        elif kind == "w8":
            x, q, s = layer
            N, K = q.shape
            w = (q.double().view(N, -1, case["gs"]) * s.double().unsqueeze(-1)).view(N, K)
            out.append(x.double() @ w.t())
        elif kind == "shared":
            x, w, d = layer
            MI = case["MI"]
            y = x.double() @ w.double().t()
            gu = _r(y[:, :2 * MI])
            g, u = gu[:, :MI], gu[:, MI:]
            sh = _r(_r(g / (1 + (-g).exp())) * u) @ d.double().t()
            res = [sh, y[:, 2 * MI:2 * MI + 1], y[:, 2 * MI + 1:]]
            if case["T"] > 4:
                res.append(_r(_r(y[:, 2 * MI:2 * MI + 1]).sigmoid()) * _r(sh))
            out.append(res)
        elif kind == "combine":
            x, wt, inv = layer
            T, k, H = case["T"], case["k"], case["H"]
            acc = torch.zeros((T, H), dtype=torch.float64, device=x.device)
            rows = inv.view(T, k)
            for j in range(k):
                acc += _r(x[rows[:, j]].double() * wt[:, j:j + 1].double())
            out.append(acc)
        else:  # the weights are whole numbers; scales are bf16(s8 * bf16(base))
            _, s8, base = layer
            out.append([None, (s8.double() * base.to(BF16).double().unsqueeze(-1)).transpose(1, 2).contiguous()])
    return out
