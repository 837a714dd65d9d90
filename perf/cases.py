"""What this package's users have it do, as measurable cases: stick-breaking attention called by itself on dense and
packed batches, and the language model built on it, evaluated and trained.  Every case goes through the public entry points
(`flame_amd.sb_attn`, `flame_amd.sb_attn_varlen`, `SBAForCausalLM`, `train_step`).

`listed()` gives the named cases, `draw()` one more of the same ranges, `prepare()` what a program holds before the call,
`run()` one pass, `work()` the least a pass can move and multiply, `tolerance()` what another correct implementation at the
same precision may differ by.
"""
import math
import random

import torch

from flame_amd import sb_attn, sb_attn_varlen
from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM
from flame_amd.train_step import make_optimizer, train_step

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
VOCAB = 32000


def listed():
    return [
        # one short sequence, as in a unit test or an interactive probe of a head: nothing but latency
        _dense("dense_tiny", B=1, H=4, T=64, D=64),
        # scoring a batch of prompts of one odd length: forward only
        _dense("dense_eval_ragged", B=4, H=16, T=1001, D=64, backward=False),
        # the operator's headline shape: one training sequence of the 340M model
        _dense("dense_train_4k", B=1, H=16, T=4096, D=64),
        # a batch in float16 with the wider heads, diagonal attended, a gradient on rem as well
        _dense("dense_train_f16_d128", B=4, H=16, T=2047, D=128, dtype="f16", attend_current=True, rem_grad=True),
        # long-context training
        _dense("dense_train_16k_d128", B=1, H=16, T=16384, D=128),
        # a float32 run, as one makes it to check a training recipe
        _dense("dense_train_f32", B=2, H=8, T=1024, D=64, dtype="f32"),
        # a large packed batch of documents of web-text lengths
        _packed("packed_train_64k", H=16, tokens=65536, D=64),
        # the 340M model's packed row, with a token count off every block edge
        _packed("packed_train_8k", H=16, tokens=8191, D=64, doc_seed=1),
        # chat turns and titles: many documents of 16 to 128 tokens
        _packed("packed_train_short_docs", H=16, tokens=65536, D=64, median=64.0, sigma=0.5, longest=128),
        # a head dim between the powers of two, fewer heads, a gradient on rem
        _packed("packed_train_d80", H=12, tokens=20011, D=80, doc_seed=2, rem_grad=True),
        # validation loss of the 340M model over a batch of equal sequences
        _model("model_eval_340m", layers=24, hidden=1024, B=2, T=2048),
        # one optimizer step of the 340M model on a packed row
        _model("model_train_340m", layers=24, hidden=1024, B=1, T=8192, train=True, packed=True),
    ]


def _dense(name, *, B, H, T, D, dtype="bf16", backward=True, attend_current=False, rem_grad=False):
    return dict(name=name, kind="dense", B=B, H=H, T=T, D=D, dtype=dtype, backward=backward,
                attend_current=attend_current, rem_grad=rem_grad)


def _packed(name, *, H, tokens, D, dtype="bf16", backward=True, attend_current=False, rem_grad=False,
            median=600.0, sigma=1.0, longest=4096, doc_seed=0):
    return dict(name=name, kind="packed", H=H, tokens=tokens, D=D, dtype=dtype, backward=backward,
                attend_current=attend_current, rem_grad=rem_grad, median=median, sigma=sigma, longest=longest,
                doc_seed=doc_seed)


def _model(name, *, layers, hidden, B, T, train=False, packed=False, doc_seed=0):
    return dict(name=name, kind="model", layers=layers, hidden=hidden, B=B, T=T, train=train, packed=packed,
                median=600.0, sigma=1.0, longest=4096, doc_seed=doc_seed)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choices(("dense", "packed", "model"), (5, 4, 2))[0]
    if kind == "model":
        hidden = rng.choice((512, 768, 1024))
        train, packed = rng.random() < 0.6, rng.random() < 0.6
        T = _log_int(rng, 256, 8192 if packed else 4096)
        B = 1 if packed else _log_int(rng, 1, max(1, 8192 // T))
        c = _model("", layers=_log_int(rng, 2, 18), hidden=hidden, B=B, T=T, train=train, packed=packed,
                   doc_seed=rng.randrange(1 << 20))
    else:
        # 16-bit types are what models train in; float32 runs stay small
        dtype = rng.choices(("bf16", "f16", "f32"), (6, 2, 1))[0]
        D = rng.choice((64, 64, 64, 128, 128, 80) if dtype == "f32" else (64, 64, 64, 128, 128, 80, 96, 256))
        H = rng.choice((1, 2, 4, 8, 12, 16, 16, 32))
        backward = rng.random() < 0.7
        opts = dict(D=D, dtype=dtype, backward=backward, attend_current=rng.random() < 0.3,
                    rem_grad=backward and rng.random() < 0.3)
        most = 16 * 16384 ** 2 * 128 // (16 if dtype == "f32" else 1)      # multiplications: the largest listed one's
        if kind == "dense":
            T = _log_int(rng, 17, 16384)
            while H * T * T * D > most:
                T = T * 7 // 10
            B = _log_int(rng, 1, max(1, min(32, most // (H * T * T * D), (1 << 21) // (H * T))))
            c = _dense("", B=B, H=H, T=T, **opts)
        else:
            longest = rng.choice((128, 1024, 4096, 4096))
            H = max(H, 4)
            tokens = _log_int(rng, 500, 65536 if dtype != "f32" else 8192)
            c = _packed("", H=H, tokens=tokens, median=min(600.0, longest / 2), sigma=0.5 if longest == 128 else 1.0,
                        longest=longest, doc_seed=rng.randrange(1 << 20), **opts)
    del c["name"]
    return c


def _doc_lengths(case, total):
    """Log-normal document lengths of 16 tokens and more that add up to `total`; the same for every seed of the values."""
    rng = random.Random(case["doc_seed"])
    lens, s = [], 0
    while s < total:
        n = round(math.exp(math.log(case["median"]) + case["sigma"] * rng.gauss(0.0, 1.0)))
        n = min(max(16, min(case["longest"], n)), total - s)
        lens.append(n)
        s += n
    return lens


def _cu_seqlens(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device="cuda")


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _qkv(case, lead, g):
    """q, k, v of shape lead + (D,) with the heads second to last but one (dense [B, H, T, D], packed [H, N, D]).  Components
    of standard deviation 0.5 as in the package's configurations; the heads differ in how far they look, as trained ones do:
    a common direction, +c in q and -c in k, moves a head's mean logit from 0 (half of the stick broken off by each key) for
    the first head to -6 (thousands of keys share it) for the last."""
    D, dtype, H = case["D"], DTYPES[case["dtype"]], case["H"]

    def rn(scale):
        return torch.randn(lead + (D,), generator=g, device="cuda") * scale

    c2 = torch.arange(H, device="cuda", dtype=torch.float32) / max(H - 1, 1) * 6.0 * math.sqrt(D)
    sign = torch.randint(0, 2, (H, D), generator=g, device="cuda") * 2.0 - 1.0
    shift = (sign * (c2 / D).sqrt()[:, None])[:, None, :]
    q = rn(0.5).add_(shift).to(dtype)
    k = rn(0.5).sub_(shift).to(dtype)
    return q, k, rn(0.5).to(dtype)


def prepare(case, seed):
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    g = _generator(seed)
    packed = case["kind"] == "packed"
    s = {"case": case}
    if packed:
        lens = _doc_lengths(case, case["tokens"])
        lead = (case["H"], case["tokens"])
        s["cu"], s["longest"] = _cu_seqlens(lens), max(lens)
    else:
        lead = (case["B"], case["H"], case["T"])
    s["qkv"] = _qkv(case, lead, g)
    if case["backward"]:
        for t in s["qkv"]:
            t.requires_grad_(True)
        dtype = DTYPES[case["dtype"]]
        s["grads"] = [torch.randn(lead + (case["D"],), generator=g, device="cuda").to(dtype)]
        if case["rem_grad"]:
            s["grads"].append(torch.randn(lead, generator=g, device="cuda").to(dtype))
    return s


def _prepare_model(case, seed):
    """The model with random weights; to train it, also its optimizer some way into a run (step count and moments as a
    checkpoint would restore them).  Weights and moments are views of one buffer each, so that run() can return them whole."""
    torch.manual_seed(seed)
    g = _generator(seed)
    cfg = SBAConfig(hidden_size=case["hidden"], num_hidden_layers=case["layers"], num_heads=case["hidden"] // 64,
                    vocab_size=VOCAB)
    with torch.device("cuda"):
        model = SBAForCausalLM(cfg)
    s = {"case": case, "model": model, "ids": torch.randint(0, VOCAB, (case["B"], case["T"]), generator=g, device="cuda")}
    s["cu"], s["longest"] = None, None
    if case["packed"]:
        lens = _doc_lengths(case, case["T"])
        s["cu"], s["longest"] = _cu_seqlens(lens), max(lens)
    if not case["train"]:
        model.eval()
        return s
    params = list(model.parameters())
    n = sum(p.numel() for p in params)
    typical = n ** -0.5                       # the gradient of one weight when the clipped norm is 1
    flat = torch.empty(n, device="cuda")
    avg = torch.randn(n, generator=g, device="cuda") * (0.2 * typical)
    avg_sq = torch.full((n,), typical * typical, device="cuda")
    opt = make_optimizer(model)
    at = 0
    for p in params:
        part = slice(at, at + p.numel())
        at = part.stop
        flat[part].copy_(p.detach().reshape(-1))
        p.data = flat[part].view(p.shape)
        opt.state[p] = {"step": torch.tensor(1000.0, device="cuda"), "exp_avg": avg[part].view(p.shape),
                        "exp_avg_sq": avg_sq[part].view(p.shape)}
    s.update(opt=opt, flat=(flat, avg, avg_sq))
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "model":
        if case["train"]:
            loss, norm = train_step(s["model"], s["opt"], s["ids"], s["ids"], s["cu"], s["longest"])
            return {"loss": loss, "norm": norm, "weights": s["flat"][0], "exp_avg": s["flat"][1], "exp_avg_sq": s["flat"][2]}
        kwargs = {} if s["cu"] is None else {"cu_seqlens": s["cu"], "max_seqlen": s["longest"]}
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            loss, logits = s["model"](s["ids"], labels=s["ids"], **kwargs)
        return {"loss": loss, "logits": logits}
    q, k, v = s["qkv"]

    def attention():
        if case["kind"] == "packed":
            return sb_attn_varlen(q, k, v, s["cu"], s["longest"], attend_current=case["attend_current"])
        return sb_attn(q, k, v, attend_current=case["attend_current"])

    if not case["backward"]:
        with torch.no_grad():
            o, rem = attention()
        return {"o": o, "rem": rem}
    o, rem = attention()
    outs = (o, rem) if case["rem_grad"] else (o,)
    dq, dk, dv = torch.autograd.grad(outs, (q, k, v), s["grads"])
    return {"o": o.detach(), "rem": rem.detach(), "dq": dq, "dk": dk, "dv": dv}


def _pairs(lens, current):
    return sum(n * (n + 1) // 2 if current else n * (n - 1) // 2 for n in lens)


def work(case):
    if case["kind"] == "model":
        cfg = SBAConfig(hidden_size=case["hidden"], num_hidden_layers=case["layers"], num_heads=case["hidden"] // 64)
        tokens = case["B"] * case["T"]
        lens = _doc_lengths(case, case["T"]) if case["packed"] else [case["T"]] * case["B"]
        block = 4 * case["hidden"] ** 2 + 3 * case["hidden"] * cfg.mlp_width()
        matrices = case["layers"] * block + case["hidden"] * VOCAB
        weights = matrices + case["hidden"] * (VOCAB + 2 * case["layers"] + 1)
        attention = 4 * case["hidden"] * _pairs(lens, False) * case["layers"]
        if case["train"]:     # weights and both moments read and written; products: forward and two of the backward
            return {"bytes": 24 * weights, "flops": 6 * matrices * tokens + 3 * attention}
        return {"bytes": 4 * weights + 2 * tokens * VOCAB, "flops": 2 * matrices * tokens + attention}
    size = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "packed":
        rows, pairs = case["H"] * case["tokens"], case["H"] * _pairs(_doc_lengths(case, case["tokens"]), case["attend_current"])
    else:
        rows = case["B"] * case["H"] * case["T"]
        pairs = case["B"] * case["H"] * _pairs([case["T"]], case["attend_current"])
    # forward: q, k, v in, o and rem out, two products of 2*D operations a pair; backward: dO (and drem) in, dq, dk, dv out,
    # four products
    tensors, vectors = (8, 1 + case["rem_grad"]) if case["backward"] else (4, 1)
    return {"bytes": size * rows * (tensors * case["D"] + vectors), "flops": (12 if case["backward"] else 4) * case["D"] * pairs}


def tolerance(case):
    if case["kind"] == "model":
        # bf16 products through every layer and, in training, back again
        return {"rel": 2e-2, "max": 0.5} if case["train"] else {"rel": 1e-2, "max": 0.2}
    return {"bf16": {"rel": 1e-2, "max": 0.3}, "f16": {"rel": 3e-3, "max": 0.1}, "f32": {"rel": 1e-5, "max": 1e-3}}[case["dtype"]]
