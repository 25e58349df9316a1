"""The work a program has this framework do, as cases that a timer can run: dense q4 / q8 projections, the MoE FFN
sublayer, the verify tail (LM head, top-k, acceptance) and the MTP draft head, each through the package's public entry
points and over the sizes they meet in use.

Sizes: d = 4096, I = 1024, 512 experts, top-10 with an FP32 router (bench.py's layer), and the served layout, d = 2560,
I = 640, a BF16 router of 513 rows and the shared expert stacked as expert 512 (11 slots a token). Token counts: 1
(decode), 2..16 (a draft's verify), tens (a short turn appended to a conversation), hundreds to 2048 (prefill chunks).
Weights are q4 G = 128 and q8 G = 64, the served groups; activations BF16, or FP32 where the engine runs in FP32.
"""
import math

import torch

from strixite_amd import ACT_BF16, ACT_F32
from strixite_amd import kernels as kx
from strixite_amd import synthetic as syn
from strixite_amd.draft import DraftHead
from strixite_amd.verify import MoeVerifyLayer, VerifyTail

E, TOPK = 512, 10


def listed():
    return [
        # One decode step's projection in the FP32 engine mode: the smallest call, launch and latency.
        linear("linear_decode_q4_f32", 4, 1, 4096, 4096, "f32", "f32"),
        # A verify of one token and five drafts through a wide q8 projection, FP32 out.
        linear("linear_verify_q8", 8, 6, 12288, 4096, "bf16", "f32"),
        # A short turn (a tool's answer, a few words) prefilled in one go: too many rows for the verify kernels.
        linear("linear_turn_q4", 4, 24, 8192, 2560, "bf16", "bf16"),
        # The same in the FP32 engine mode, which keeps the activations' 24 bits, through a q8 projection.
        linear("linear_turn_q8_f32", 8, 37, 2560, 4096, "f32", "f32"),
        # The ragged last chunk of a prompt through a q4 projection.
        linear("linear_prefill_q4", 4, 1531, 7680, 2560, "bf16", "bf16"),
        # The MoE sublayer of one decode step: ten experts' weights.
        moe("moe_decode", "wide", 1, 0.0),
        # The MoE sublayer of a six-token verify.
        moe("moe_verify", "wide", 6, 0.0),
        # The same verify in the served layout: BF16 router, shared expert, 66 slots.
        moe("moe_verify_served", "served", 6, 0.0),
        # A short prompt's MoE sublayer in the served layout: few tokens an expert, nearly every expert hit.
        moe("moe_prompt_served", "served", 200, 0.0),
        # A full prefill chunk, experts chosen with a Zipf skew (0 to some 400 rows an expert).
        moe("moe_prefill", "wide", 2048, 0.3),
        # The end of a six-token verify: q8 LM head, top-40 of each row, sampled acceptance of five drafts.
        tail("tail_verify", 6, 151936, 4096, 40, "sampled"),
        # One MTP draft: the q4 copy of the head's first 65,536 rows and the pick.
        {"name": "draft_head", "kind": "draft", "V": 65536, "K": 4096},
    ]


def linear(name, bits, M, N, K, act, out):
    return {"name": name, "kind": "linear", "bits": bits, "M": M, "N": N, "K": K, "act": act, "out": out}


def moe(name, layout, M, skew):
    return {"name": name, "kind": "moe", "layout": layout, "M": M, "skew": skew}


def tail(name, M, V, K, kc, mode):
    return {"name": name, "kind": "tail", "M": M, "V": V, "K": K, "kc": kc, "mode": mode}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["moe"] * 4 + ["tail", "draft"])
    if kind == "linear":
        bits = rng.choice([4, 8])
        act = rng.choice(["bf16", "bf16", "bf16", "f32"])
        # the FP32 engine mode runs decode, verify and short turns
        M = _log_int(rng, 1, 2048 if act == "bf16" else 128)
        N = rng.choice([_log_int(rng, 300, 14000), 16 * _log_int(rng, 20, 800), 256 * rng.randint(2, 48)])
        K = rng.choice([1024, 2048, 2560, 4096, 128 * rng.randint(4, 32)])
        case = linear("", bits, M, N, K, act, "f32" if act == "f32" else rng.choice(["bf16", "f32"]))
    elif kind == "moe":
        M = _log_int(rng, 1, 2000)
        case = moe("", rng.choice(["wide", "served"]), M, rng.choice([0.0, 0.3]) if M >= 64 else 0.0)
    elif kind == "tail":
        case = tail("", rng.randint(1, 16), rng.choice([151936, 8 * rng.randint(4000, 31000)]), rng.choice([2560, 4096]),
                    rng.randint(20, 64), rng.choice(["greedy", "sampled"]))
    else:
        case = {"kind": "draft", "V": 64 * _log_int(rng, 128, 1024), "K": rng.choice([2560, 4096])}
    case.pop("name", None)
    return case


# ---- inputs ----

def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _dims(case):
    """d, I, slots a token, experts in the weights."""
    return (4096, 1024, TOPK, E) if case["layout"] == "wide" else (2560, 640, TOPK + 1, E + 1)


def _act(case):
    return torch.float32 if case["act"] == "f32" else torch.bfloat16


class ServedLayer:
    """The served MoE sublayer as a program strings it together: BF16 router with the shared gate in row E, the shared
    expert stacked as expert E. Up to five tokens go slot by slot, more are grouped by expert."""

    def __init__(self, Wr, gate_up, down, M):
        dev, A, d, I = Wr.device, TOPK + 1, gate_up.K, down.K
        self.Wr, self.gate_up, self.down, self.M, self.A = Wr, gate_up, down, M, A
        self.logits = torch.empty((M, E + 1), dtype=torch.float32, device=dev)
        self.ids = torch.empty((M, A), dtype=torch.int32, device=dev)
        self.coef = torch.empty((M, A), dtype=torch.float32, device=dev)
        self.err = torch.zeros(4, dtype=torch.int32, device=dev)
        self.ws = torch.empty(kx.route_workspace_bytes(M, A, E + 1) // 4, dtype=torch.int32, device=dev)
        self.h = torch.empty((M, A, I), dtype=torch.bfloat16, device=dev)
        self.partial = torch.empty((M * A, d), dtype=torch.float32, device=dev)
        self.y = torch.empty((M, d), dtype=torch.bfloat16, device=dev)

    def forward(self, x):
        kx.linear_bf16w(x, self.Wr, out_act=ACT_F32, y=self.logits)
        kx.moe_router(self.logits, E, TOPK, shared=self.logits[:, E:], shared_ld=E + 1, shared_id=E, ids=self.ids,
                      coef=self.coef, err=self.err)
        if self.M < 6:
            kx.experts_gather(x, self.gate_up, E + 1, self.ids, swiglu=True, y=self.h, err=self.err)
            kx.experts_combine(self.h, self.down, E + 1, self.ids, self.coef, y=self.y, err=self.err)
        else:
            kx.group_routes(self.ids, E + 1, ws=self.ws, err=self.err)
            kx.gather_grouped(x, self.gate_up, E + 1, self.ws, self.M, self.A, swiglu=True, y=self.h)
            kx.combine_grouped(self.h, self.down, E + 1, self.ids, self.coef, self.ws, partial=self.partial, y=self.y)
        return self.y


def _moe_inputs(case, seed):
    d, I, _, Ew = _dims(case)
    x = syn.activations(case["M"], d, seed=seed)
    Wr = syn.router_weight(E if case["layout"] == "wide" else E + 1, d, seed=seed + 1)
    if case["skew"] > 0:  # the skew as a bias on a constant channel of x
        x[:, 0] = 1.0
        Wr[:E, 0] = syn.zipf_router_bias(E, seed=seed + 2, scale=case["skew"])
    if case["layout"] == "served":
        Wr = Wr.to(torch.bfloat16)
    return x, Wr, syn.qweight(4, Ew * 2 * I, d, 128, seed=seed + 3), syn.qweight(4, Ew * d, I, 128, seed=seed + 4)


def _drafts(h, head, case, seed):
    """Draft tokens as a draft head proposes them: each row's most likely token, up to a row drawn from the seed and
    another token from there on; and the host's uniform draws."""
    g = _gen(seed, "cpu")
    k = case["M"] - 1
    best = _rows_times(h.float(), head, torch.float32).argmax(1).to(torch.int32)[:k]
    off = torch.arange(k) >= int(torch.randint(0, k + 1, (1,), generator=g))
    best = torch.where(off.to(best.device), (best + 1) % case["V"], best)
    u = torch.rand(k + 1, dtype=torch.float64, generator=g).cuda()
    return best.contiguous(), u


def prepare(case, seed):
    seed = 1000 * seed + 17
    if case["kind"] == "linear":
        G = 128 if case["bits"] == 4 else 64
        w = syn.qweight(case["bits"], case["N"], case["K"], G, seed=seed)
        x = syn.activations(case["M"], case["K"], seed=seed + 1, dtype=_act(case))
        y = torch.empty((case["M"], case["N"]), dtype=torch.float32 if case["out"] == "f32" else torch.bfloat16,
                        device="cuda")
        return {"case": case, "w": w, "x": x, "y": y}
    if case["kind"] == "moe":
        x, Wr, gu, dn = _moe_inputs(case, seed)
        if case["layout"] == "wide":
            layer = MoeVerifyLayer(Wr, gu, dn, E, TOPK, case["M"])
        else:
            layer = ServedLayer(Wr, gu, dn, case["M"])
        return {"case": case, "x": x, "layer": layer}
    if case["kind"] == "tail":
        head = syn.qweight(8, case["V"], case["K"], 64, seed=seed)
        h = syn.activations(case["M"], case["K"], seed=seed + 1)
        drafts, u = _drafts(h, head, case, seed + 2)
        t = VerifyTail(head, case["V"], case["kc"], case["M"])
        t.out.fill_(-1)
        return {"case": case, "h": h, "drafts": drafts, "u": u, "tail": t}
    head = DraftHead(syn.qweight(8, case["V"], case["K"], 64, seed=seed), case["V"])
    return {"case": case, "h": syn.activations(1, case["K"], seed=seed + 1), "head": head}


def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        out = ACT_F32 if case["out"] == "f32" else ACT_BF16
        return kx.linear(state["x"], state["w"], out_act=out, y=state["y"])
    if case["kind"] == "moe":
        layer = state["layer"]
        y = layer.forward(state["x"])
        return {"y": y, "logits": layer.logits, "ids": layer.ids, "coef": layer.coef}
    if case["kind"] == "tail":
        t = state["tail"]
        temperature = 0.0 if case["mode"] == "greedy" else 0.7
        out = t.forward(state["h"], state["drafts"], state["u"], temperature, 20, 0.95)
        return {"out": out, "logits": t.logits, "values": t.cands[..., 0].view(torch.float32),
                "tokens": t.cands[..., 1], "nan": t.nan}
    pick = state["head"].forward(state["h"])
    return {"logits": state["head"].logits, "best": pick[:4].view(torch.int32),
            "values": pick[4:12].view(torch.float32), "flags": pick[12:].view(torch.int32)}


# ---- what a pass cannot do without ----

def _qbytes(bits, N, K, G):
    return N * (K * bits // 8 + 4 * (K // G))


def work(case):
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        size = {"f32": 4, "bf16": 2}
        return {"bytes": _qbytes(case["bits"], N, K, 128 if case["bits"] == 4 else 64) + M * K * size[case["act"]] +
                M * N * size[case["out"]], "flops": 2 * M * N * K}
    if case["kind"] == "moe":
        M = case["M"]
        d, I, A, Ew = _dims(case)
        hit = E * (1 - (1 - TOPK / E) ** M) + (A - TOPK)  # distinct experts, uniformly routed
        router = E * d * 4 if case["layout"] == "wide" else (E + 1) * d * 2
        expert = _qbytes(4, 2 * I, d, 128) + _qbytes(4, d, I, 128)
        return {"bytes": round(hit * expert) + router + 2 * M * d * 2 + M * Ew * 4 + M * A * 8,
                "flops": 2 * M * A * 3 * I * d + 2 * M * Ew * d}
    M, V, K = case.get("M", 1), case["V"], case["K"]
    head = _qbytes(8, V, K, 64) if case["kind"] == "tail" else _qbytes(4, V, K, 64)
    return {"bytes": head + M * K * 2 + M * V * 4, "flops": 2 * M * V * K}


def tolerance(case):
    """About four times the error against `exact`: FP32 sums (q4 codes enter as 128 + code, whose cancellation costs a
    few bits, more of them with FP32 activations), or the BF16 rounding of the outputs."""
    if case["kind"] == "linear":
        if case["out"] == "bf16":
            return {"rel": 7e-3}
        return {"rel": 2e-6 if case["bits"] == 8 else 2e-5 if case["act"] == "f32" else 6e-6}
    if case["kind"] == "moe":
        # two logits within FP32 rounding of each other may swap places, or swap an expert
        return {"rel": 1.4e-2, "differ": max(1e-3, 4 / (case["M"] * _dims(case)[2]))}
    if case["kind"] == "tail":
        return {"rel": 2e-6, "differ": max(1e-3, 2 / (case["M"] * case["kc"]))}
    return {"rel": 4e-6}


# ---- the same results in 64 bits ----

def _dequant(w, r0, r1, dtype=torch.float64):
    """Rows [r0, r1) of a quantized weight as code * scale + min."""
    n, per, groups = r1 - r0, w.K * w.bits // 8, w.K // w.G
    q = w.q[r0 * per:r1 * per].view(n, per)
    if w.bits == 4:
        q = torch.stack((q & 15, q >> 4), dim=2).view(n, w.K)
    s = w.scale[r0 * groups:r1 * groups].view(torch.bfloat16).view(n, groups, 1).to(dtype)
    m = w.minv[r0 * groups:r1 * groups].view(torch.bfloat16).view(n, groups, 1).to(dtype)
    return (q.view(n, groups, w.G).to(dtype) * s + m).view(n, w.K)


def _rows_times(x, w, dtype=torch.float64):
    """x [M, K] times the weight's rows, a few thousand rows at a time."""
    x = x.to(dtype)
    return torch.cat([x @ _dequant(w, r, min(r + 8192, w.N), dtype).T for r in range(0, w.N, 8192)], dim=1)


def _best(scores, k):
    """The k largest of each row, larger first and the lower index first among equals: values and indices."""
    v, i = torch.sort(scores, dim=1, descending=True, stable=True)
    return v[:, :k], i[:, :k].to(torch.int32)


def _exact_moe(case, seed):
    x, Wr, gu, dn = _moe_inputs(case, seed)
    d, I, _, _ = _dims(case)
    x64 = x.double()
    logits = x64 @ Wr.double().T
    top, ids = _best(logits[:, :E], TOPK)
    coef = torch.softmax(top, dim=1)
    if case["layout"] == "served":
        ids = torch.cat([ids, torch.full_like(ids[:, :1], E)], dim=1)
        coef = torch.cat([coef, torch.sigmoid(logits[:, E:])], dim=1)
    y = torch.zeros(case["M"], d, dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        rows, slot = torch.nonzero(ids == e, as_tuple=True)
        gate, up = (x64[rows] @ _dequant(gu, 2 * I * e, 2 * I * (e + 1)).T).split(I, dim=1)
        out = (torch.nn.functional.silu(gate) * up) @ _dequant(dn, d * e, d * (e + 1)).T
        y.index_add_(0, rows, coef[rows, slot][:, None] * out)
    return {"y": y, "logits": logits, "ids": ids, "coef": coef}


def exact(case, seed):
    if case["kind"] == "moe":
        return _exact_moe(case, 1000 * seed + 17)
    state = prepare(case, seed)
    if case["kind"] == "linear":
        return _rows_times(state["x"], state["w"])
    if case["kind"] == "tail":
        logits = _rows_times(state["h"], state["tail"].w)
        values, tokens = _best(logits, case["kc"])
        return {"out": None, "logits": logits, "values": values, "tokens": tokens, "nan": None}
    logits = _rows_times(state["h"], state["head"].w)
    values, tokens = _best(logits, 2)
    return {"logits": logits, "best": tokens[0, :1], "values": values[0], "flags": None}
