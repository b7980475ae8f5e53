"""The sampling stage's workloads for timing and comparison: single calls through the package's public entry points, from one
greedy row to a batch of 256 rows at the full vocabulary (V = 248,320), over the ranges that `draw` spans.

Kinds of case:
  step     Sampler.run over rows packed once (PackedBatch), the batch loop's call.  hist > 0: the rows' generated tokens,
           in ProcState slots (state) or passed with the call; advance: the call also takes the decode step on the device.
  graph    the same call and StepBook.finish captured in one HIP graph, which the decode loop replays.
  request  Sampler.sample over RowSpecs: the call that packs the rows itself, as a server without state slots makes it.
  verify   Sampler.verify: K drafts of each of B sequences against their K + 1 target rows.
  draft    Sampler.draft_pick: the drafter's picks over its reduced vocabulary, with the draft probabilities.
  head     HeadSelect: the R best candidates of a quantised head's logits, rescored from the bf16 head.

Logits: "chat" is N(0, 2.5) with 32 ids 8 higher (a model that knows a few continuations), "wide" N(0, 3) (every outlier
its own), "flat" N(0, 0.5) (a nucleus of most of the vocabulary)."""
import math

import numpy as np
import torch

import qwen_warp_amd as q

DEV = "cuda"
V = 248320
BASE = dict(kind="step", B=1, V=V, dtype="float32", logits="chat", temperature=1.0, top_k=0, top_p=1.0, min_p=0.0, hist=0, state=False, advance=False,
            repetition=1.0, presence=0.0, frequency=0.0, bias=0, banned=False, stop=0, mixed=False)


def _case(**kw):
    return {**BASE, **kw}


def listed():
    return [
        # one row, greedy, no processors: the smallest call, all launch latency
        _case(name="greedy_1", dtype="bfloat16", temperature=0.0),
        # one user's chat decode step (top-k 20, top-p 0.8, repetition 1.05 over 2,048 tokens), replayed from a graph with its bookkeeping
        _case(name="graph_1", kind="graph", temperature=0.7, top_k=20, top_p=0.8, repetition=1.05, hist=2048, state=True),
        # eight users, each with parameters and a history (512 to 32,768 tokens) of their own, passed with the call
        _case(name="mixed_8", B=8, dtype="bfloat16", hist=32768, mixed=True),
        # sixteen requests handed over as they came from the server: the rows packed in the call
        _case(name="request_16", kind="request", B=16, dtype="bfloat16", temperature=0.8, top_p=0.95, presence=0.5, frequency=0.3, hist=1500),
        # 300 biases, three suppressed stop tokens and a banned mask on every row, top-k 50
        _case(name="bias_32", B=32, dtype="bfloat16", logits="wide", temperature=0.6, top_k=50, bias=300, banned=True, stop=3),
        # a server's batch of chat rows: mixed parameters, state slots, the step taken on the device
        _case(name="chat_64", B=64, dtype="bfloat16", hist=4096, mixed=True, state=True, advance=True),
        # near-flat rows, top-p 0.95 (a nucleus of ~200,000 tokens), repetition 1.1 over 4,096 tokens, the step taken on the device
        _case(name="flat_64", B=64, logits="flat", top_p=0.95, repetition=1.1, hist=4096, state=True, advance=True),
        # the widest batch: no processors, top-p 0.95
        _case(name="wide_256", B=256, logits="wide", top_p=0.95),
        # speculative verify, 8 drafts of 4 sequences (36 target rows), a drafter of its own mind: mostly rejections
        _case(name="verify_4x8", kind="verify", B=4, K=8, Vd=64000, logits="wide", top_p=0.95, aligned=False),
        # 4 drafts of 16 sequences, a drafter that follows the target, penalties from state slots, top-k / top-p
        _case(name="verify_16x4", kind="verify", B=16, K=4, Vd=64000, dtype="bfloat16", temperature=0.8, top_k=50, top_p=0.95, repetition=1.1, hist=4096,
              state=True, aligned=True),
        # one draft step of 16 sequences: the picks and their distributions over a drafter's 64,000 ids
        _case(name="draft_16", kind="draft", B=16, V=64000, temperature=0.8, top_k=20, top_p=0.95),
        # the quantised head's 64 best of each of 16 positions, rescored
        _case(name="head_16", kind="head", B=16, K=5120, R=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step", "graph", "request", "verify", "verify", "draft", "head"))
    c = dict(BASE, kind=kind, dtype=rng.choice(("float32", "bfloat16")), logits=rng.choice(("chat", "chat", "wide", "flat")),
             V=8 * rng.choice((V // 8, _log(rng, 4000, 32768))))
    if kind == "head":
        return dict(c, dtype="float32", B=rng.randint(1, 16), V=4 * _log(rng, 8000, V // 4), K=8 * _log(rng, 128, 640), R=rng.choice((8, 20, 40, 64)))
    c.update(temperature=round(rng.uniform(0.3, 1.2), 2), top_k=rng.choice((0, 0, 20, 50, 1000)), top_p=rng.choice((1.0, 0.8, 0.95, round(rng.uniform(0.5, 1.0), 3))))
    if kind == "draft":
        return dict(c, B=_log(rng, 1, 32), V=8 * _log(rng, 2000, 16000))
    c.update(min_p=rng.choice((0.0, 0.0, 0.05)), repetition=rng.choice((1.0, 1.1)), presence=rng.choice((0.0, 0.5)), frequency=rng.choice((0.0, 0.3)))
    if c["repetition"] != 1.0 or c["presence"] or c["frequency"]:
        c.update(hist=_log(rng, 100, 16384), state=kind != "request" and rng.random() < 0.6)
    if kind == "verify":
        return dict(c, B=_log(rng, 1, 16), K=rng.randint(1, 8), Vd=8 * _log(rng, 1000, 8000), aligned=rng.random() < 0.5)
    if rng.random() < 0.25:
        c.update(bias=_log(rng, 8, 1000), banned=rng.random() < 0.5, stop=rng.choice((0, 3)))
    if kind == "step":
        return dict(c, B=_log(rng, 1, 256), advance=c["state"] and rng.random() < 0.7, mixed=rng.random() < 0.3, temperature=rng.choice((0.0, c["temperature"], c["temperature"], c["temperature"])))
    if kind == "graph":
        return dict(c, B=_log(rng, 1, 16), state=True, hist=max(c["hist"], 100))
    B = _log(rng, 1, 16)  # request
    return dict(c, B=B, hist=min(c["hist"], 24000 // B), bias=min(c["bias"], 64))


# ------------------------------------------------------------------------------------------ inputs
def _logits(g, rows, c):
    x = torch.randn(rows, c["V"], device=DEV, generator=g)
    if c["logits"] == "chat":
        x = x.mul_(2.5)
        ids = torch.randint(0, c["V"], (rows, 32), device=DEV, generator=g)
        x.scatter_add_(1, ids, torch.full(ids.shape, 8.0, device=DEV))
    else:
        x = x.mul_(0.5 if c["logits"] == "flat" else 3.0)
    return x.to(getattr(torch, c["dtype"]))


def _history(r, n, vocab):
    """n ids whose frequencies fall with their rank (Zipf, s = 1), the ranks scattered over the vocabulary."""
    rank = np.exp(r.random(n) * math.log(vocab)).astype(np.int64)
    return (rank * 104729 + 12345) % vocab


def _rows(c, r, n=None):
    """(n or B) RowSpecs with their generated tokens in `gen`."""
    rows = []
    for b in range(n or c["B"]):
        d = {k: c[k] for k in ("temperature", "top_k", "top_p", "min_p", "repetition", "presence", "frequency")}
        hist = c["hist"]
        if c["mixed"]:
            d.update(temperature=float(np.round(0.3 + 0.9 * r.random(), 2)), top_k=(0, 20, 50, 1000)[b % 4], top_p=float(np.round(0.5 + 0.5 * r.random(), 3)),
                     min_p=float(np.round(0.1 * r.random(), 3)), presence=float(np.round(1.5 * r.random(), 2)), frequency=float(np.round(1.5 * r.random(), 2)))
            hist >>= b % 7  # 32,768 down to 512 where hist is 32,768
        bias = None
        if c["bias"]:
            ids = r.choice(c["V"], c["bias"], replace=False)
            bias = dict(zip(ids.tolist(), (200.0 * r.random(c["bias"]) - 100.0).tolist()))
        banned = None
        if c["banned"]:  # one token in 128
            w = np.full((c["V"] + 31) // 32, 0xFFFFFFFF, np.uint32)
            for _ in range(7):
                w &= r.integers(0, 1 << 32, w.size, dtype=np.uint32)
            banned = w
        gen = _history(r, hist, c["V"])
        rows.append(q.RowSpec(**d, bias=bias, banned=banned, gen=gen.tolist() if c["kind"] == "request" else gen, min_tokens=hist + 1 if c["stop"] else 0,
                              stop=[c["V"] - 3 - 2 * k for k in range(c["stop"])], seed=int(r.integers(1 << 62)), position=int(r.integers(1 << 20)), row_key=b))
    return rows


def _into_slots(rows, vocab):
    """The rows with their generated tokens in the slots of a ProcState."""
    state = q.ProcState(len(rows), vocab, DEV)
    for b, row in enumerate(rows):
        state.begin(b, (), row.gen)
        row.ngen, row.gen, row.state_slot = len(row.gen), (), b
    return state


def prepare(case, seed):
    c, kind = case, case["kind"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = np.random.default_rng(seed)
    if kind == "head":
        w = torch.randn(c["V"], c["K"], device=DEV, generator=g, dtype=torch.bfloat16).mul_(0.02)
        x = torch.randn(c["B"], c["K"], device=DEV, generator=g).to(torch.bfloat16)
        approx = (x @ w.t()).float()
        approx += 0.05 * torch.randn(approx.shape, device=DEV, generator=g)  # what the quantised head is off by
        return dict(kind=kind, select=q.HeadSelect(DEV), w=w, x=x, logits=approx.contiguous(), R=c["R"])
    s = dict(kind=kind, sampler=q.Sampler(DEV))
    if kind == "draft":
        s["rows"] = [q.draft_row(temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"], seed=int(r.integers(1 << 62)), j=1 + b % 8,
                                 position=int(r.integers(1 << 20)), row_key=b) for b in range(c["B"])]
        s["logits"] = _logits(g, c["B"], c)
        s["idmap"] = torch.randperm(4 * c["V"], device=DEV, generator=g)[:c["V"]].to(torch.int32)
        return s
    rows = _rows(c, r)
    if kind == "request":
        return dict(s, rows=rows, logits=_logits(g, c["B"], c))
    state = _into_slots(rows, c["V"]) if c["state"] else None
    if kind == "verify":
        target = _logits(g, c["B"] * (c["K"] + 1), c).view(c["B"], c["K"] + 1, c["V"])
        idmap = torch.randperm(c["V"], device=DEV, generator=g)[:min(c["Vd"], c["V"])].to(torch.int32)
        draft = torch.randn(c["B"], c["K"], idmap.numel(), device=DEV, generator=g)
        draft = draft + target[:, :c["K"]].float()[:, :, idmap.long()] if c["aligned"] else 3.0 * draft
        probs = torch.softmax(draft, dim=2)
        pick = (probs / torch.empty_like(probs).exponential_(generator=g)).argmax(2)
        drafts = idmap[pick].contiguous()
        packed = q.PackedBatch(q.Sampler.verify_rows(rows, drafts.tolist()), c["V"], DEV, state)
        return dict(s, target=target, probs=probs, inv=s["sampler"].verify_map(idmap, c["V"]), drafts=drafts, rows=rows, packed=packed, state=state)
    s.update(state=state, packed=q.PackedBatch(rows, c["V"], DEV, state), logits=_logits(g, c["B"], c), advance=c["advance"])
    if kind == "graph":
        s["tokens"] = torch.empty(c["B"], dtype=torch.int32, device=DEV)
        s["book"] = book = q.StepBook(c["B"], device=DEV)
        for b in range(c["B"]):
            book.start(b, 0, -1)
        s["seqs"] = torch.arange(c["B"], dtype=torch.int32, device=DEV)
        s["sampler"].run(s["packed"], s["logits"], out_tokens=s["tokens"])
        torch.cuda.synchronize()
        s["graph"], side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.cuda.graph(s["graph"], stream=side):
            s["sampler"].run(s["packed"], s["logits"], out_tokens=s["tokens"])
            book.finish(s["seqs"], s["tokens"], state=state, rows=s["packed"])
        torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------------------------------ one pass
def run(state):
    s, kind = state, state["kind"]
    if kind == "step":
        tokens = s["sampler"].run(s["packed"], s["logits"], advance=s["advance"])
        return [tokens, s["packed"].rows_t] if s["advance"] else tokens  # the rows as the step leaves them
    if kind == "graph":
        s["graph"].replay()
        return s["tokens"], s["book"].seqs, s["book"].rings, s["packed"].rows_t
    if kind == "request":
        return s["sampler"].sample(s["logits"], s["rows"])
    if kind == "verify":
        return s["sampler"].verify(s["target"], s["probs"], s["inv"], s["drafts"], s["rows"], packed=s["packed"])
    if kind == "draft":
        return s["sampler"].draft_pick(s["logits"], s["rows"], s["idmap"])
    return [*s["select"](s["logits"], s["w"], s["x"], s["R"]), s["logits"]]


def work(case):
    c, kind = case, case["kind"]
    size = 4 if c["dtype"] == "float32" else 2
    if kind == "head":
        return dict(bytes=4 * c["B"] * c["V"] + c["B"] * c["R"] * (2 * c["K"] + 12) + 2 * c["B"] * c["K"], flops=2 * c["B"] * c["R"] * c["K"])
    rows = c["B"] * (c["K"] + 1 if kind == "verify" else 1)
    hist = sum(c["hist"] >> b % 7 for b in range(c["B"])) if c["mixed"] else c["B"] * c["hist"]
    n = rows * c["V"] * size + 4 * hist + c["B"] * (8 * c["bias"] + 4 * c["stop"] + (c["V"] // 8 if c["banned"] else 0)) + 4 * rows
    if kind == "verify":
        n += 4 * c["B"] * c["K"] * min(c["Vd"], c["V"]) + 4 * min(c["Vd"], c["V"]) + 4 * c["B"] * (c["K"] + 1)
    if kind == "draft":
        n += 4 * c["B"] * c["V"] + 8 * c["B"]
    # the weight of a token: the scaling, the exponent's floor and fraction, one multiply-add, one add to a sum
    return dict(bytes=n, flops=6 * rows * c["V"] if c["temperature"] > 0 else 0)


def tolerance(case):
    if case["kind"] == "draft":
        return {"rel": 2e-6}  # weights of 24 bits, x / T in fp32 (1.7e-7 from 64 bits as measured; x / T rounded otherwise moves 5e-7)
    if case["kind"] == "head":
        return {"rel": 4e-7}  # fp32 sums of K exact bf16 products (4.9e-8 from 64 bits as measured; another order about 1e-7)
    return "exact"  # tokens are defined bit for bit (integer weights, Philox draws)


def exact(case, seed):
    c = case
    if c["kind"] == "draft":
        s = prepare(c, seed)
        z = s["logits"].double() / float(np.float32(c["temperature"]))
        z, order = torch.sort(z, dim=1, descending=True, stable=True)
        if c["top_k"]:
            z[:, c["top_k"]:] = -math.inf
        p = torch.softmax(z, dim=1)
        before = p.cumsum(1) - p
        if c["top_p"] < 1.0:
            p = torch.where(before < float(np.float32(c["top_p"])), p, torch.zeros_like(p))
        p = p / p.sum(1, keepdim=True)
        return None, torch.zeros_like(p).scatter_(1, order, p), None
    if c["kind"] == "head":
        s = prepare(c, seed)
        cand = torch.sort(s["logits"], dim=1, descending=True, stable=True).indices[:, :c["R"]]
        val = torch.stack([s["w"][cand[t]].double() @ s["x"][t].double() for t in range(c["B"])])
        return None, val.max(1).values, None, val, s["logits"].double().scatter(1, cand, val)
    return None  # tokens: no 64-bit value
