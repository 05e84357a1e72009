"""The sampler's work in real use, as cases that can be timed and compared: decode steps of one
row up to 1,024 rows over vocabularies of 32,000 to 262,144 logits, greedy, top-k, nucleus (top-k off),
min-p and per-request parameters, with and without a repetition penalty, and the LM head's product
with and without the pick.

A case is a dict of plain values: `call` names the entry point, the rest its sizes, its sampling
parameters and how its logits are distributed. listed() holds the named ones, draw(rng) gives more of
the same ranges.
"""
import math

import numpy as np
import torch

import verbo_amd
from verbo_amd import decode

SAMPLED = dict(temp=0.8, top_k=0, top_p=1.0, min_p=0.0, repeat=1.0, hist=0)


def _case(name, call, rows, vocab, **kw):
    c = dict(name=name, call=call, rows=rows, vocab=vocab, logits="model", bf16=False, **SAMPLED)
    c.update(kw)
    return c


def listed():
    return [
        # one chat session decoding: the reference's default top-k 40 on a 49,152-token model
        _case("decode_topk_1x49152", "pick", 1, 49152, logits="spiky", temp=0.7, top_k=40, top_p=0.9, repeat=1.1, hist=64),
        # one chat session decoding with nucleus sampling only (top-k off), a large vocabulary
        _case("decode_nucleus_1x151936", "pick", 1, 151936, top_p=0.95, repeat=1.1, hist=512),
        # the drop-in verbo::Sampler's pick: the row is in host memory
        _case("host_pick_1x49152", "host", 1, 49152, logits="spiky", temp=0.7, top_k=40, top_p=0.9, repeat=1.1, hist=64),
        # a small server batch on nucleus + min-p, logits of a model that computes them in bf16 (ties)
        _case("nucleus_16x128256_bf16", "pick", 16, 128256, logits="spiky", bf16=True, temp=1.0, top_p=0.95, min_p=0.02),
        # one step of a continuous-batching server: 24 live slots of requests with their own parameters
        _case("serve_24x50257", "serve", 24, 50257, logits="spiky"),
        # a medium server batch on a chat model's recommended options
        _case("topk_32x151936", "pick", 32, 151936, temp=0.7, top_k=20, top_p=0.8, repeat=1.05, hist=256),
        # greedy decoding of 64 rows with a penalty
        _case("greedy_64x151936", "pick", 64, 151936, logits="spiky", temp=0.0, repeat=1.15, hist=256),
        # the benchmark's batch: every stage of the sampler on 256 rows
        _case("topk_256x151936", "pick", 256, 151936, temp=0.8, top_k=50, top_p=0.95, min_p=0.05, repeat=1.1, hist=512),
        # nucleus sampling of a large batch with nearly flat rows (high-temperature rollouts)
        _case("nucleus_512x151936_flat", "pick", 512, 151936, logits="flat", temp=1.0, top_p=0.99),
        # a large server batch, every row with its own parameters and history
        _case("mixed_1024x128256", "mixed", 1024, 128256, logits="spiky", hist=2048),
        # the LM head and the pick in one call, a decode batch
        _case("head_pick_64x151936x896", "head_pick", 64, 151936, hidden=896, temp=0.8, top_k=50, top_p=0.95, min_p=0.05,
              repeat=1.1, hist=512),
        # the LM head alone, a large decode batch (or the scored positions of a prompt)
        _case("head_logits_256x151936x896", "head_logits", 256, 151936, hidden=896),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["pick"] * 9 + ["host", "serve", "serve", "mixed", "head_pick", "head_pick", "head_logits"])
    vocab = rng.choice([49152, 128256, 151936, 50257, _log_int(rng, 32000, 262144), _log_int(rng, 32000, 262144) | 1])
    if call.startswith("head"):
        vocab = min(vocab, 151936)
        hidden = 64 * rng.randint(8, 14)
        c = dict(call=call, rows=_log_int(rng, 1, 256), vocab=vocab, logits="model", bf16=False, **SAMPLED, hidden=hidden)
        if call == "head_pick":
            c.update(temp=round(rng.uniform(0.5, 1.2), 2), top_k=rng.choice([20, 40, 50, 100]), top_p=round(rng.uniform(0.8, 1.0), 2),
                     repeat=1.1, hist=_log_int(rng, 16, 1024))
        return c
    logits, bf16 = rng.choice(["model", "spiky", "flat"]), rng.random() < 0.3
    c = dict(call=call, rows=1, vocab=vocab, logits=logits, bf16=bf16, **SAMPLED)
    if call == "serve":
        c["rows"] = _log_int(rng, 2, 128)
        return c
    if call == "mixed":
        c.update(rows=min(_log_int(rng, 8, 1024), 1024 * 128256 // vocab), logits=rng.choice(["model", "spiky"]), hist=_log_int(rng, 16, 2048))
        return c
    c["temp"] = round(rng.uniform(0.3, 1.5), 2)
    if rng.random() < 0.6:
        c.update(repeat=round(rng.uniform(1.0, 1.3), 2), hist=_log_int(rng, 16, 2048))
    kind = rng.choice(["topk", "topk", "nucleus", "nucleus", "nucleus", "greedy"])
    if kind == "topk":
        c.update(top_k=rng.choice([1, 10, 20, 40, 50, 100, 256, 400, 1000]), top_p=round(rng.uniform(0.7, 1.0), 2))
    elif kind == "nucleus":
        c.update(top_p=round(rng.uniform(0.5, 1.0), 2))
    else:
        c.update(temp=0.0)
    if kind != "greedy" and rng.random() < 0.4:
        c.update(min_p=rng.choice([0.01, 0.02, 0.05, 0.1]))
    if call == "pick":  # up to the largest listed batch; rows that the general path takes cost more each
        c["rows"] = min(_log_int(rng, 1, 512), 512 * 151936 // vocab)
    return c


# ---- inputs -----------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _logits(case, seed):
    """[rows, vocab] fp32 on the GPU, rows padded to 16 bytes. model: a Gumbel bulk with some 2,000 raised
    tokens, most of the mass on few of them; spiky: a normal bulk with 16 tokens far above it; flat:
    N(0, 0.5^2)."""
    g, B, V = _gen(seed), case["rows"], case["vocab"]
    x = torch.empty(B, (V + 3) // 4 * 4, device="cuda")
    if case["logits"] == "model":
        x.exponential_(generator=g).clamp_(min=1e-30).log_().mul_(-2.0)
        ids = torch.randint(V, (B, 2000), generator=g, device="cuda")
        x.scatter_add_(1, ids, (12.0 * torch.arange(1, 2001, device="cuda") ** -1.1).expand(B, 2000))
    elif case["logits"] == "spiky":
        x.normal_(0.0, 2.0, generator=g)
        ids = torch.randint(V, (B, 16), generator=g, device="cuda")
        x.scatter_add_(1, ids, 4.0 + 6.0 * torch.rand(B, 16, generator=g, device="cuda"))
    else:
        x.normal_(0.0, 0.5, generator=g)
    if case["bf16"]:
        x = x.bfloat16().float()
    return x[:, :V]


def _hist(case, seed, logits):
    """CSR histories: per row `hist` ids, half of them among its 64 largest logits (what was said already
    is likely again), the rest anywhere."""
    B, V, H = case["rows"], case["vocab"], case["hist"]
    if H == 0:
        return None, None
    g = _gen(seed + 1)
    ids = torch.randint(V, (B, H), generator=g, device="cuda")
    if logits is not None:
        top = logits.topk(min(64, V), dim=1).indices
        ids[:, : H // 2] = top.gather(1, torch.randint(top.shape[1], (B, H // 2), generator=g, device="cuda"))
    off = torch.arange(B + 1, dtype=torch.int32, device="cuda") * H
    return ids.to(torch.int32).reshape(-1).contiguous(), off


def _fields(case, seed):
    return dict(temp=case["temp"], top_k=case["top_k"], top_p=case["top_p"], min_p=case["min_p"], repeat=case["repeat"],
                repeat_last=0, seed=seed)


def _row_fields(case, seed, repeat_last):
    """Parameters of requests that ask for different things: a quarter greedy, a quarter with top-k off."""
    r = np.random.RandomState(seed & 0x7FFFFFFF)
    rows = []
    for i in range(case["rows"]):
        rows.append(dict(temp=0.0 if r.rand() < 0.25 else float(np.float32(0.05 + 1.45 * r.rand())), top_k=int(r.choice([0, 20, 40, 100])),
                         top_p=float(np.float32(0.8 + 0.2 * r.rand())), min_p=float(r.choice([0.0, 0.05, 0.1])),
                         repeat=float(np.float32(1.0 + 0.3 * r.rand())), repeat_last=repeat_last, seed=1000 + seed % 100000 * 1024 + i))
    return rows


def _prompts(case, seed):
    r = np.random.RandomState((seed + 2) & 0x7FFFFFFF)
    return [r.randint(0, case["vocab"], size=r.randint(8, 200)).astype(np.int32) for _ in range(case["rows"])]


def prepare(case, seed):
    s = {"call": case["call"], "ctx": verbo_amd.Context(0)}
    if case["call"] in ("head_pick", "head_logits"):
        g, D = _gen(seed), case["hidden"]
        s["hidden"] = torch.randn(case["rows"], D, generator=g, device="cuda").bfloat16()
        s["head"] = (torch.randn(case["vocab"], D, generator=g, device="cuda") * (2.5 / D ** 0.5)).bfloat16()
        if case["call"] == "head_pick":
            s["params"] = verbo_amd.Params(**_fields(case, seed))
            s["hist"], s["off"] = _hist(case, seed, None)
        return s
    logits = _logits(case, seed)
    if case["call"] == "host":
        s["logits"] = logits[0].cpu().numpy().copy()
        s["params"] = verbo_amd.Params(**_fields(case, seed))
        hist, _ = _hist(case, seed, logits)
        s["hist"] = hist.cpu().numpy() if hist is not None else np.zeros(0, np.int32)
        s["u"] = float(np.random.RandomState(seed & 0x7FFFFFFF).rand())
        return s
    s["logits"] = logits
    if case["call"] == "serve":  # a decoder with some more slots than are live, the live ones spread over them
        rows = _row_fields(case, seed, 64)
        s["dec"] = decode.BatchDecoder.with_slots(case["rows"] + 8, case["vocab"])
        s["stream"] = torch.cuda.current_stream()
        slots = sorted(np.random.RandomState(seed & 0x7FFFFFFF).permutation(case["rows"] + 8)[: case["rows"]].tolist())
        for slot, p, ids in zip(slots, rows, _prompts(case, seed)):
            s["dec"].admit(slot, verbo_amd.Params(**p), ids, s["stream"])
        s["rows"] = torch.tensor(slots, dtype=torch.int32, device="cuda")
        s["active"] = torch.ones(case["rows"], dtype=torch.int32, device="cuda")
        s["out"] = torch.empty(case["rows"], dtype=torch.int32, device="cuda")
        return s
    if case["call"] == "mixed":
        s["params"] = verbo_amd.to_device_params(verbo_amd.params_array(_row_fields(case, seed, 0)))
    else:
        s["params"] = verbo_amd.Params(**_fields(case, seed))
    s["hist"], s["off"] = _hist(case, seed, logits)
    return s


def run(s):
    call = s["call"]
    if call == "host":
        return s["ctx"].pick_host(s["logits"], s["params"], s["hist"], s["u"])
    if call == "head_logits":
        return s["ctx"].head_logits(s["hidden"], s["head"])
    if call == "head_pick":
        return s["ctx"].head_pick(s["hidden"], s["head"], s["params"], s["hist"], s["off"])
    if call == "serve":
        s["dec"].pick_rows(s["logits"], s["rows"], s["out"], s["stream"])
        s["dec"].accept_rows(s["out"], s["rows"], s["active"], s["stream"])
        return s["out"]
    return s["ctx"].pick_batch(s["logits"], s["params"], s["hist"], s["off"])


def work(case):
    B, V, H = case["rows"], case["vocab"], case["hist"]
    if case["call"] == "head_logits":
        D = case["hidden"]
        return {"bytes": 2 * D * (B + V) + 4 * B * V, "flops": 2 * B * V * D}
    if case["call"] == "head_pick":
        D = case["hidden"]
        return {"bytes": 2 * D * (B + V) + 4 * B * H + 4 * B, "flops": 2 * B * V * D}
    return {"bytes": 4 * B * V + 4 * B * H + 4 * B + (32 * B if case["call"] in ("mixed", "serve") else 0), "flops": 0}


def tolerance(case):
    # the logits: 32-bit sums of exact bf16 products; another order of the same sums lies 2.7e-7 (2-norm) and
    # 3.0e-6 (largest) away
    return {"rel": 1.1e-6, "max": 1.2e-5} if case["call"] == "head_logits" else "exact"


# ---- the same results in 64 bits ----------------------------------------------------------------------

_M64 = (1 << 64) - 1


def _splitmix(state):
    z = state = (state + 0x9E3779B97F4A7C15) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return state, z ^ (z >> 31)


def _draw_counter(seed):
    return (_splitmix(seed)[1] >> 11) * 2.0 ** -53


def _draw_stream(seed):
    """The first draw of a request's xorshift128+ stream (its output is taken before the update)."""
    state, a = _splitmix(seed)
    b = _splitmix(state)[1]
    return (((a + b) & _M64) >> 11) * 2.0 ** -53


def _pick64(row, p, window, u):
    """One pick from a GPU row: penalty, order (value descending, index ascending), top-k, min-p, top-p, draw."""
    v = row.clone()
    f32 = lambda x: torch.tensor(x, dtype=torch.float32, device=v.device)  # noqa: E731
    if p["repeat"] != 1.0 and window is not None and window.numel():
        ids = window.long().unique()
        ids = ids[(ids >= 0) & (ids < v.numel())]
        x = v[ids]
        v[ids] = torch.where(x > 0, x / f32(p["repeat"]), x * f32(p["repeat"]))
    if p["temp"] <= 0.0:
        return int((v == v.max()).nonzero()[0])
    order = torch.sort(v, descending=True, stable=True)
    k = p["top_k"] if 0 < p["top_k"] < v.numel() else v.numel()
    val, idx = order.values[:k], order.indices[:k]
    pr = torch.exp((val - val[0]).double() / float(np.float32(p["temp"]))).cpu().numpy()
    total = pr.cumsum()[-1]
    keep = k
    if p["min_p"] > 0.0:
        low = np.nonzero(pr < pr[0] * float(np.float32(p["min_p"])))[0]
        keep = max(1, int(low[0])) if low.size else k
    top_p = float(np.float32(p["top_p"]))
    if 0.0 < top_p < 1.0:
        over = np.nonzero((pr[:keep] / total).cumsum() >= top_p)[0]
        keep = int(over[0]) + 1 if over.size else keep
    cdf = pr[:keep].cumsum()
    at = np.nonzero(cdf >= u * cdf[-1])[0]
    return int(idx[int(at[0]) if at.size else keep - 1])


def exact(case, seed):
    s = prepare(case, seed)
    call, B, H = case["call"], case["rows"], case["hist"]
    if call in ("head_logits", "head_pick"):
        parts = [s["hidden"].double() @ w.double().t() for w in s["head"].split(16384)]
        logits = torch.cat(parts, 1)
        if call == "head_logits":
            return logits
        logits = logits.float()
    elif call == "host":
        h = torch.from_numpy(s["hist"]).cuda()
        return _pick64(torch.from_numpy(s["logits"]).cuda(), _fields(case, seed), h, s["u"])
    else:
        logits = s["logits"]
    ids = []
    rows = _row_fields(case, seed, 64 if call == "serve" else 0) if call in ("mixed", "serve") else None
    prompts = _prompts(case, seed) if call == "serve" else None
    for r in range(B):
        if call == "serve":
            p = rows[r]
            ids.append(_pick64(logits[r], p, torch.from_numpy(prompts[r][-64:]).cuda(), _draw_stream(p["seed"])))
            continue
        p = rows[r] if rows else _fields(case, seed)
        window = s["hist"][r * H:(r + 1) * H] if H else None
        ids.append(_pick64(logits[r], p, window, _draw_counter(p["seed"] if rows else p["seed"] + r)))
    return torch.tensor(ids, dtype=torch.int32)
