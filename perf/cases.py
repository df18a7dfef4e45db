"""The calls whose speed counts, and how to make, run and check them.

Four kinds of work, each through the entry point a program calls:

decode   a decode step: fused_moe.decode_layer (gate, selection, permutation,
         experts, combine) of several layers, captured once and replayed, each
         layer with its own weights, slot table and hidden states.  Layers
         whose routed experts exceed the bank run the overflow pass from a
         stage buffer.
experts  one layer's experts over given routing, eager, every expert resident:
         fused_moe.fused_experts, as a prefill chunk runs them.
waves    one layer's prefill past its bank, the waves planned on the device and
         staged from page-locked host memory: fused_moe.run_device_waves.
router   gate and expert selection of a prefill chunk: fused_moe.route.

Weights are N(0, 0.02), hidden states N(0, 1), all bf16.  "skew" scales a
Zipf(1.1) rank bias on the routing logits (1: ranks mapped onto [-2, 2]; 0:
none).  Decode inputs are drawn so that no token's selection hangs on the
rounding of a logit (the k-th score leads the next by a few bf16 steps): then
the routing, and so the output, is the same for every correct router.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "vllm-ascend-hust-latchmoe_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

# The layer shapes of the benchmark and the tests: experts E, hidden H,
# expert width I, experts per token k; S pinned shared experts of the routed
# shape appended to every token; groups: grouped sigmoid scores with a
# selection bias (8 groups, 4 kept, x 2.5), else softmax.
SHAPES = {
    "qwen3": dict(E=128, H=2048, I=768, k=8, S=0, groups=0),
    "qwen1.5": dict(E=60, H=2048, I=1408, k=4, S=0, groups=0),
    "deepseek": dict(E=256, H=7168, I=2048, k=8, S=1, groups=8),
}
TOPK_GROUP, ROUTED_SCALE = 4, 2.5


def listed():
    return [
        # one user's token: the smallest step, launches and latency count
        dict(name="decode-1", kind="decode", shape="qwen3", tokens=1, layers=8, slots=64, skew=1.0),
        # a few concurrent users
        dict(name="decode-4", kind="decode", shape="qwen3", tokens=4, layers=8, slots=64, skew=1.0),
        # an ordinary serving batch
        dict(name="decode-16", kind="decode", shape="qwen3", tokens=16, layers=6, slots=64, skew=1.0),
        # a large batch whose experts exceed the 64-slot bank
        dict(name="decode-64-overflow", kind="decode", shape="qwen3", tokens=64, layers=3, slots=64, skew=1.0),
        # a large odd batch, every expert resident, routing without a bias
        dict(name="decode-111", kind="decode", shape="qwen3", tokens=111, layers=2, slots=128, skew=0.0),
        # a layer of wider experts whose width is no multiple of 256 columns
        dict(name="decode-24-wide", kind="decode", shape="qwen1.5", tokens=24, layers=3, slots=60, skew=0.5),
        # the 88 MB experts, grouped router and pinned shared expert
        dict(name="decode-8-deepseek", kind="decode", shape="deepseek", tokens=8, layers=1, slots=256, skew=0.0),
        # a chunk of a chunked prefill (or a prompt of ordinary length)
        dict(name="chunk-300", kind="experts", shape="qwen3", tokens=300, skew=0.5),
        # a long prefill with every expert resident
        dict(name="prefill-4096", kind="experts", shape="qwen3", tokens=4096, skew=0.0),
        # the same for the 88 MB experts: few tokens per expert
        dict(name="prefill-2048-deepseek", kind="experts", shape="deepseek", tokens=2048, skew=0.0),
        # a long prefill with the experts in host memory
        dict(name="prefill-4096-staged", kind="waves", shape="qwen3", tokens=4096, slots=48, skew=0.0),
        # routing of a long prefill
        dict(name="route-4096", kind="router", shape="qwen3", tokens=4096, skew=0.5),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choices(["decode", "experts", "router", "waves"], [10, 7, 2, 1])[0]
    skew = round(rng.choice([0.0, 1.0, rng.uniform(0.0, 1.2)]), 3)
    if kind == "waves":
        return dict(kind=kind, shape="qwen3", tokens=_log_int(rng, 400, 4096), slots=rng.randint(32, 64), skew=skew)
    shape = rng.choices(["qwen3", "qwen1.5", "deepseek"], [6, 2, 2])[0]
    E = SHAPES[shape]["E"]
    if kind == "router":
        return dict(kind=kind, shape=shape, tokens=_log_int(rng, 65, 4096), skew=skew)
    if kind == "experts":
        return dict(kind=kind, shape=shape, tokens=_log_int(rng, 20, 2048 if shape == "deepseek" else 4096), skew=skew)
    tokens = _log_int(rng, 1, 32 if shape == "deepseek" else 128)
    layers = 1 if shape == "deepseek" else 8 if tokens <= 8 else 4 if tokens <= 32 else 2
    slots = E if shape == "deepseek" else rng.choice([64, 96, E]) if shape == "qwen3" else rng.choice([40, E])
    return dict(kind=kind, shape=shape, tokens=tokens, layers=layers, slots=slots, skew=skew)


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + part)


def _normal(shape, g, std=0.02):
    t = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    return t.normal_(0.0, std, generator=g)


def _rank_bias(case, seed, part):
    """Zipf(1.1) over a random rank of the experts, mapped onto [-2, 2] and
    scaled by the case's skew."""
    E = SHAPES[case["shape"]]["E"]
    ranks = np.random.RandomState((int(seed) * 31 + part) % (1 << 31)).permutation(E) + 1
    logp = -1.1 * np.log(ranks.astype(np.float64))
    lo = -1.1 * math.log(E)
    return torch.from_numpy((case["skew"] * (-2.0 + 4.0 * (logp - lo) / -lo)).astype(np.float32)).cuda()


def _choice_scores(logits, bias, sh):
    """(selection scores, weight scores), f64, of bf16 logits."""
    if not sh["groups"]:
        z = logits + bias
        return z, torch.softmax(z, dim=1)
    s = torch.sigmoid(logits)
    return s + bias, s


def _top(score, k):
    """Ids of the k largest, the lower id first among equals."""
    return torch.sort(score, dim=1, descending=True, stable=True)[1][:, :k]


def _select(logits, bias, sh):
    """(ids, f64 weights, margin) of f64 logits that are rounded to bf16
    here; margin: the smallest lead of what is selected (experts, and groups
    where there are any) over what is not."""
    z = logits.to(torch.bfloat16).double()
    choice, score = _choice_scores(z, bias.double(), sh)
    k = sh["k"]
    margin = torch.full((z.shape[0],), math.inf, dtype=torch.float64, device=z.device)
    if sh["groups"]:
        T, G = z.shape[0], sh["groups"]
        per = choice.view(T, G, -1)
        g2 = per.topk(2, dim=2)[0].sum(2)
        gs = torch.sort(g2, dim=1, descending=True)[0]
        margin = gs[:, TOPK_GROUP - 1] - gs[:, TOPK_GROUP]
        keep = torch.zeros_like(g2, dtype=torch.bool).scatter_(1, _top(g2, TOPK_GROUP), True)
        choice = choice.masked_fill(~keep.unsqueeze(2).expand_as(per).reshape(T, -1), -math.inf)
    ids = _top(choice, k)
    s = torch.sort(choice, dim=1, descending=True)[0]
    margin = torch.minimum(margin, s[:, k - 1] - s[:, k])
    w = score.gather(1, ids)
    w = w / w.sum(1, keepdim=True) * (ROUTED_SCALE if sh["groups"] else 1.0)
    return ids, w, margin


def _with_shared(ids, w, sh):
    if not sh["S"]:
        return ids, w
    T = ids.shape[0]
    suffix = torch.arange(sh["E"], sh["E"] + sh["S"], device=ids.device, dtype=ids.dtype).expand(T, sh["S"])
    return torch.cat([ids, suffix], 1), torch.cat([w, torch.ones((T, sh["S"]), dtype=w.dtype, device=w.device)], 1)


def _decode_inputs(case, seed, layer):
    """One decode layer: gate weight, bias, hidden states and their routing."""
    sh, T = SHAPES[case["shape"]], case["tokens"]
    g = _gen(seed, 16 * layer)
    gate = _normal((sh["E"], sh["H"]), g)
    # grouped scores: a small selection bias beside the sigmoid scores
    bias = _normal((sh["E"],), g, 0.01).float() if sh["groups"] else _rank_bias(case, seed, layer)
    cand = _normal((8 * T + 64, sh["H"]), g, 1.0)
    margin = _select(cand.double() @ gate.double().t(), bias, sh)[2]
    sure = margin > (0.004 if sh["groups"] else 0.03)
    rows = torch.sort((~sure).to(torch.int8), stable=True)[1][:T]
    x = cand[rows].contiguous()
    ids, w, _ = _select(x.double() @ gate.double().t(), bias, sh)
    ids, w = _with_shared(ids, w, sh)
    return gate, bias, x, ids, w


def _bank(n, sh, g):
    return _normal((n, 2 * sh["I"], sh["H"]), g), _normal((n, sh["H"], sh["I"]), g)


def _tables(case, seed, layer, ids):
    """Slot tables of the bank and of the overflow buffer: the routed experts
    (all of them where the bank holds every expert) at random slots, the
    shared experts in the pinned suffix; what the bank cannot hold is in the
    overflow buffer, and in no bank slot."""
    sh, P = SHAPES[case["shape"]], case["slots"]
    r = np.random.RandomState((int(seed) * 131 + layer) % (1 << 31))
    used = np.arange(sh["E"]) if P >= sh["E"] else np.unique(ids[:, : sh["k"]].cpu().numpy())
    used = r.permutation(used)
    table = np.full(sh["E"] + sh["S"], -1, dtype=np.int32)
    table[used[:P]] = r.permutation(P)[: min(P, used.size)]
    table[sh["E"]:] = P + np.arange(sh["S"])
    rest = used[P:]
    over = np.full_like(table, -1)
    over[rest] = np.arange(rest.size)
    return table, over, rest.size


def _experts_inputs(case, seed):
    """Hidden states and routing of a prefill: logits of unit spread (what a
    trained gate gives) plus the rank bias, then the shape's selection."""
    sh, T = SHAPES[case["shape"]], case["tokens"]
    g = _gen(seed, 1)
    x = _normal((T, sh["H"]), g, 1.0)
    bias = _rank_bias(case, seed, 3)
    logits = torch.randn((T, sh["E"]), generator=g, device="cuda").double()
    if sh["groups"]:
        ids, w, _ = _select(logits + bias, torch.zeros_like(bias), sh)
    else:
        ids, w, _ = _select(logits, bias, sh)
    ids, w = _with_shared(ids, w, sh)
    table = np.random.RandomState(int(seed) % (1 << 31)).permutation(sh["E"] + sh["S"]).astype(np.int32)
    return x, ids.to(torch.int32).contiguous(), w.to(torch.bfloat16).contiguous(), torch.from_numpy(table).cuda()


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _router_spec(case, bias):
    from vllm_moe_offload_amd import fused_moe

    sh = SHAPES[case["shape"]]
    if sh["groups"]:
        return fused_moe.RouterSpec(top_k=sh["k"], scoring_func="sigmoid", use_grouped_topk=True,
                                    num_expert_group=sh["groups"], topk_group=TOPK_GROUP,
                                    routed_scaling_factor=ROUTED_SCALE, e_score_correction_bias=bias, n_shared=sh["S"])
    return fused_moe.RouterSpec(top_k=sh["k"], logit_bias=bias)


def _prepare_decode(case, seed):
    from vllm_moe_offload_amd import fused_moe
    from vllm_moe_offload_amd.moe_offload.slot_mapping import PreparedSlotWeights

    sh, T, P = SHAPES[case["shape"]], case["tokens"], case["slots"]
    kw, n_slots = sh["k"] + sh["S"], P + sh["S"]
    layers, outs = [], []
    for l in range(case["layers"]):
        gate, bias, x, ids, _ = _decode_inputs(case, seed, l)
        table, over, n_over = _tables(case, seed, l, ids)
        w13, w2 = _bank(n_slots, sh, _gen(seed, 16 * l + 1))
        overflow = None
        if n_over:
            o13, o2 = _bank(P, sh, _gen(seed, 16 * l + 2))
            overflow = PreparedSlotWeights(w1=o13, w2=o2, log2phy=torch.from_numpy(over).cuda(),
                                           physical_expert_count=P, mapping=None)
        layers.append(dict(x=x, gate=gate, spec=_router_spec(case, bias), w13=w13, w2=w2,
                           table=torch.from_numpy(table).cuda(), overflow=overflow))
        dev = dict(device="cuda")
        outs.append(dict(out=torch.zeros((T, sh["H"]), dtype=torch.bfloat16, **dev),
                         logits=torch.zeros((T, sh["E"]), dtype=torch.bfloat16, **dev),
                         weights=torch.zeros((T, kw), dtype=torch.bfloat16, **dev),
                         ids=torch.zeros((T, kw), dtype=torch.int32, **dev)))
    ws = fused_moe.get_workspace(T, kw, n_slots, sh["H"], sh["I"], "cuda", tag="perf")

    def step():
        for a, o in zip(layers, outs):
            fused_moe.decode_layer(a["x"], a["gate"], a["spec"], a["w13"], a["w2"], a["table"], workspace=ws,
                                   out=o["out"], logits_out=o["logits"], w_out=o["weights"], ids_out=o["ids"],
                                   overflow=a["overflow"])

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return dict(kind="decode", graph=graph, layers=layers, outs=outs, ws=ws)


def _prepare_waves(case, seed):
    from vllm_moe_offload_amd.moe_offload.config import MoeOffloadConfig
    from vllm_moe_offload_amd.moe_offload.runtime import MoeOffloadRuntime

    sh = SHAPES[case["shape"]]
    x, ids, w, _ = _experts_inputs(case, seed)
    w13, w2 = _bank(sh["E"], sh, _gen(seed, 2))
    host = []
    for t in (w13, w2):
        h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
        h.copy_(t)
        host.append(h)
    del w13, w2
    rt = MoeOffloadRuntime(MoeOffloadConfig(enabled=True, num_slots=case["slots"], async_load=True,
                                            b2_wave_prefill=True, device_wave_prefill=True))
    rt.register_host_buffers(layer_id=0, w13_host=host[0], w2_host=host[1], slot_device=torch.device("cuda"))
    return dict(kind="waves", rt=rt, x=x, ids=ids, w=w, E=sh["E"], out=torch.zeros_like(x))


def prepare(case, seed):
    sh, T = SHAPES[case["shape"]], case["tokens"]
    if case["kind"] == "decode":
        return _prepare_decode(case, seed)
    if case["kind"] == "waves":
        return _prepare_waves(case, seed)
    if case["kind"] == "router":
        g = _gen(seed, 1)
        x, gate = _normal((T, sh["H"]), g, 1.0), _normal((sh["E"], sh["H"]), g)
        bias = _normal((sh["E"],), g, 0.01).float() if sh["groups"] else _rank_bias(case, seed, 3)
        kw = sh["k"] + sh["S"]
        return dict(kind="router", x=x, gate=gate, spec=_router_spec(case, bias),
                    logits=torch.zeros((T, sh["E"]), dtype=torch.bfloat16, device="cuda"),
                    w=torch.zeros((T, kw), dtype=torch.bfloat16, device="cuda"),
                    ids=torch.zeros((T, kw), dtype=torch.int32, device="cuda"))
    x, ids, w, table = _experts_inputs(case, seed)
    w13, w2 = _bank(sh["E"] + sh["S"], sh, _gen(seed, 2))
    return dict(kind="experts", x=x, ids=ids, w=w, table=table, w13=w13, w2=w2, out=torch.zeros_like(x))


def run(state):
    from vllm_moe_offload_amd import fused_moe

    s = state
    if s["kind"] == "decode":
        s["graph"].replay()
        return s["outs"]
    if s["kind"] == "router":
        w, ids, logits = fused_moe.route(s["x"], s["gate"], s["spec"], logits_out=s["logits"], w_out=s["w"],
                                         ids_out=s["ids"])
        return dict(logits=logits, weights=w, ids=ids)
    if s["kind"] == "waves":
        return fused_moe.run_device_waves(s["rt"], layer_id=0, hidden=s["x"], topk_weights=s["w"],
                                          topk_ids=s["ids"], num_logical_experts=s["E"], out=s["out"])
    return fused_moe.fused_experts(s["x"], s["w"], s["ids"], s["w13"], s["w2"], s["table"], out=s["out"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, how close outputs must be, and their values
# ---------------------------------------------------------------------------
def _distinct(case):
    """Experts that one layer's tokens select, by simulation."""
    sh, T = SHAPES[case["shape"]], case["tokens"]
    r = np.random.RandomState(7)
    got = []
    for _ in range(3):
        ranks = r.permutation(sh["E"]) + 1
        logp = -1.1 * np.log(ranks.astype(np.float64))
        lo = -1.1 * math.log(sh["E"])
        spread = 0.02 * math.sqrt(sh["H"]) if case["kind"] in ("decode", "router") else 1.0
        z = spread * r.standard_normal((T, sh["E"])) + case["skew"] * (-2.0 + 4.0 * (logp - lo) / -lo)
        if sh["groups"]:
            per = z.reshape(T, sh["groups"], -1)
            s2 = np.sort(1 / (1 + np.exp(-per)), axis=2)[:, :, -2:].sum(2)
            cut = np.sort(s2, axis=1)[:, -TOPK_GROUP][:, None]
            z = np.where((s2 >= cut)[:, :, None], per, -np.inf).reshape(T, -1)
        got.append(np.unique(np.argpartition(-z, sh["k"] - 1, axis=1)[:, : sh["k"]]).size)
    return sum(got) / len(got) + sh["S"]


def work(case):
    sh, T = SHAPES[case["shape"]], case["tokens"]
    kw, expert = sh["k"] + sh["S"], 3 * sh["H"] * sh["I"] * 2
    router = dict(bytes=sh["E"] * sh["H"] * 2 + T * (2 * sh["E"] + 6 * kw), flops=2 * T * sh["H"] * sh["E"])
    if case["kind"] == "router":
        return dict(bytes=router["bytes"] + T * sh["H"] * 2, flops=router["flops"])
    one = dict(bytes=_distinct(case) * expert + 2 * T * sh["H"] * 2 + T * kw * 6, flops=6 * T * kw * sh["H"] * sh["I"])
    if case["kind"] == "decode":
        return {n: case["layers"] * (one[n] + router[n]) for n in one}
    return one


def tolerance(case):
    # bf16 act, expert rows and output: the path is 2e-3 to 4e-3 off its
    # value in 64 bits (three roundings of 2^-9 each, relative, over a sum of
    # k expert rows); logits one bf16 step; a selection between scores that
    # are equal in bf16 may fall on the other one
    if case["kind"] == "router":
        return {"rel": 1e-2, "max": 0.25, "differ": 5e-3}
    return {"rel": 1e-2, "max": 6e-2, "differ": 0.0}


def _expert_sum(x, ids, w, slots, banks, H):
    """sum_j w[t, j] * down(silu(gate) * up) in 64 bits; slots[e]: (bank,
    slot) of expert e."""
    out = torch.zeros((x.shape[0], H), dtype=torch.float64, device="cuda")
    xd = x.double()
    for e in torch.unique(ids).tolist():
        b, s = slots[e]
        t, j = torch.nonzero(ids == e, as_tuple=True)
        gu = xd[t] @ banks[b][0][s].double().t()
        I = gu.shape[1] // 2
        act = gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]
        out.index_add_(0, t, (act @ banks[b][1][s].double().t()) * w[t, j].double().unsqueeze(1))
    return out


def exact(case, seed):
    sh = SHAPES[case["shape"]]
    if case["kind"] == "router":
        g = _gen(seed, 1)
        x, gate = _normal((case["tokens"], sh["H"]), g, 1.0), _normal((sh["E"], sh["H"]), g)
        bias = _normal((sh["E"],), g, 0.01).float() if sh["groups"] else _rank_bias(case, seed, 3)
        logits = x.double() @ gate.double().t()
        ids, w = _with_shared(*_select(logits, bias, sh)[:2], sh)
        # the weights of a token whose selection hangs on a rounding have no such value
        return dict(logits=logits, weights=None, ids=None)
    if case["kind"] == "decode":
        got = []
        for l in range(case["layers"]):
            gate, bias, x, ids, w = _decode_inputs(case, seed, l)
            table, over, n_over = _tables(case, seed, l, ids)
            banks = [_bank(case["slots"] + sh["S"], sh, _gen(seed, 16 * l + 1))]
            if n_over:
                banks.append(_bank(case["slots"], sh, _gen(seed, 16 * l + 2)))
            slots = {e: (0, int(table[e])) if table[e] >= 0 else (1, int(over[e])) for e in range(table.size)}
            got.append(dict(out=_expert_sum(x, ids, w.to(torch.bfloat16), slots, banks, sh["H"]),
                            logits=x.double() @ gate.double().t(), weights=w, ids=None))
        return got
    x, ids, w, table = _experts_inputs(case, seed)
    banks = [_bank(sh["E"] + sh["S"], sh, _gen(seed, 2))]
    place = range(sh["E"] + sh["S"]) if case["kind"] == "waves" else table.tolist()
    return _expert_sum(x, ids, w, {e: (0, s) for e, s in enumerate(place)}, banks, sh["H"])
