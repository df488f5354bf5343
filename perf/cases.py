"""The engine's work in use, as cases a timing program can run and check.

A case goes through the package's public entry points (autoresearch_amd.engine)
on the two model shapes the repository serves: the depth-12 model (d_model 768,
6 heads of 128) and the depth-20 model with two grouped KV heads (d_model 1280,
10 heads of 128), both with a vocabulary of 8192. Six kinds of call:

  forward   forward_dev on device buffers: logits and, with targets, the
            per-token cross-entropy (prefill; split-bf16 or fp16 operands)
  eval      eval_bpb over rows of host ids (the bits-per-byte run)
  prompt    a prompt through step_multi in chunks into a KV cache, then one
            step for the logits of its last id (the way to the first token)
  decode    decode_greedy from a filled cache, with every step's logits
  sample    decode_sample (nucleus, penalties, 3-gram ban) from a filled
            cache, then one step over the last id for its logits
  step      one cached step on host buffers (gpt_step as an app calls it)

Weights are N(0, 0.02) like the repository's seeded ones, except lm_head: its
rows are N(0, 0.08) plus a multiple of another id's embedding, so that every
id has a likely successor and next-id distributions are peaked as a trained
model's are (greedy ids then do not hang on ties in the last bit).
"""
import math

import numpy as np
import torch

from autoresearch_amd import engine
from autoresearch_amd.weights import Dims

SHAPES = {  # n_layer, d_model, n_head, n_kv_head, head_dim, vocab
    "d12": (12, 768, 6, 6, 128, 8192),
    "gqa20": (20, 1280, 10, 2, 128, 8192),
}
EPS = 1e-5
LAYER_STACKS = ("c_q", "c_k", "c_v", "c_proj", "c_fc", "c_proj2")


def listed():
    return [
        # the headline prefill: one full context, logits and cross-entropy
        dict(name="forward_f16_2048", kind="forward", model="d12", B=1, T=2048, f16=True, nll=True),
        # the same call in the default operand format, ragged rows
        dict(name="forward_split_2x777", kind="forward", model="d12", B=2, T=777, f16=False, nll=False),
        # a short prefill, where launches and latency count
        dict(name="forward_f16_150", kind="forward", model="d12", B=1, T=150, f16=True, nll=True),
        # the bits-per-byte run at its usual batch of full rows
        dict(name="eval_f16_8x2048", kind="eval", model="d12", rows=8, T=2048, batch=8, f16=True),
        # a chat prompt in chunks of 64, as the app feeds it
        dict(name="prompt_d12_500", kind="prompt", model="d12", P=500, chunk=64, kv16=False),
        # a long prompt of the grouped-KV model in one pass
        dict(name="prompt_gqa20_1791", kind="prompt", model="gqa20", P=1791, chunk=2048, kv16=False),
        # chat: one sequence, greedy
        dict(name="decode_d12_b1", kind="decode", model="d12", B=1, ctx=300, steps=32, kv16=False),
        dict(name="decode_gqa20_b1", kind="decode", model="gqa20", B=1, ctx=1500, steps=16, kv16=False),
        # batched serving: a few sequences on the default cache, many on the bf16 one
        dict(name="decode_d12_b7", kind="decode", model="d12", B=7, ctx=260, steps=16, kv16=False),
        dict(name="decode_d12_b64_kv16", kind="decode", model="d12", B=64, ctx=1024, steps=8, kv16=True),
        # chat with sampling
        dict(name="sample_d12", kind="sample", model="d12", ctx=120, steps=24),
        # the smallest call: one step on host buffers
        dict(name="step_d12_b1", kind="step", model="d12", B=1, ctx=64, kv16=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "eval", "prompt", "prompt", "decode", "decode",
                       "decode", "sample", "step"])
    if kind == "forward":
        model = rng.choice(["d12", "d12", "d12", "gqa20"])
        B = rng.choice([1, 1, 1, 2, 3, 4])
        return dict(kind=kind, model=model, B=B, T=_log_int(rng, 6, 2048 // B),
                    f16=rng.random() < 0.5, nll=rng.random() < 0.5)
    if kind == "eval":
        rows = rng.randint(1, 8)
        f16 = rng.random() < 0.5
        return dict(kind=kind, model="d12", rows=rows, T=_log_int(rng, 64, 2048 if f16 else 1200),
                    batch=rng.randint(1, rows), f16=f16)
    if kind == "prompt":
        model = rng.choice(["d12", "d12", "d12", "gqa20"])
        chunk = rng.choice([16, 64, 64, 128, 2048])
        most = min(2047, chunk * (8 if model == "d12" else 4))
        return dict(kind=kind, model=model, P=_log_int(rng, 20, most), chunk=chunk,
                    kv16=rng.random() < 0.3)
    if kind == "decode":
        model = rng.choice(["d12", "d12", "d12", "gqa20"])
        B = rng.choice([1, _log_int(rng, 2, 64), _log_int(rng, 5, 64)])
        most = 4 if B > 16 else (32 if B == 1 else 10) // (1 if model == "d12" else 3)
        return dict(kind=kind, model=model, B=B, ctx=_log_int(rng, 16, 2000 if B <= 16 else 1024),
                    steps=rng.randint(2, most), kv16=rng.random() < 0.4)
    if kind == "sample":
        return dict(kind=kind, model="d12", ctx=_log_int(rng, 8, 1500), steps=rng.randint(4, 40))
    return dict(kind=kind, model=rng.choice(["d12", "d12", "gqa20"]), B=rng.choice([1, 1, 2, 4, 6]),
                ctx=_log_int(rng, 8, 1500), kv16=rng.random() < 0.3)


# ------------------------------------------------------------------ inputs

def _dims(case):
    L, D, H, KH, hd, V = SHAPES[case["model"]]
    return Dims(n_layer=L, d_model=D, n_head=H, n_kv_head=KH, head_dim=hd, vocab=V, eps=EPS)


def _weights(case, seed):
    """The eight stacked tensors, bf16-representable fp32 values, on the GPU."""
    L, D, H, KH, hd, V = SHAPES[case["model"]]
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)

    def normal(n, std):
        t = torch.randn(n, generator=g, device="cuda", dtype=torch.float32).mul_(std)
        return t.to(torch.bfloat16).float()

    q, k = H * hd * D, KH * hd * D
    w = {"wte": normal(V * D, 0.02)}
    for name, n in zip(LAYER_STACKS, (q, k, k, q, 4 * D * D, 4 * D * D)):
        w[name] = normal(L * n, 0.02)
    nxt = torch.randperm(V, generator=g, device="cuda")
    lm = torch.randn(V, D, generator=g, device="cuda", dtype=torch.float32).mul_(0.08)
    lm[nxt] += 2.5 * w["wte"].view(V, D)
    w["lm_head"] = lm.to(torch.bfloat16).float().view(-1)
    return w


def _rope(n, hd):
    """Host fp32 tables (n, hd/2), as an app builds them."""
    theta = np.power(np.float32(10000.0), np.float32(-2.0) * np.arange(hd // 2, dtype=np.float32)
                     / np.float32(hd)).astype(np.float32)
    ang = (np.arange(n, dtype=np.float32)[:, None] * theta[None, :]).astype(np.float32)
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _ids(case, seed):
    """Host ids [B, n] of the case (targets one position on, in forward and eval)."""
    V = SHAPES[case["model"]][5]
    B, n = _rows(case)
    p = np.arange(1, V + 1, dtype=np.float64) ** -1.1  # ranks of a Zipf law, shuffled over ids
    r = np.random.default_rng(seed)
    return r.permutation(V)[r.choice(V, size=(B, n), p=p / p.sum())].astype(np.int32)


def _rows(case):
    k = case["kind"]
    if k == "forward":
        return case["B"], case["T"] + 1
    if k == "eval":
        return case["rows"], case["T"] + 1
    if k == "prompt":
        return 1, case["P"]
    return case.get("B", 1), case["ctx"] + 1


def _token_bytes(seed, V):
    return np.random.default_rng(seed + 7).integers(0, 9, V).astype(np.int32)


SAMPLING = dict(temp=0.8, topp=0.9, pres=0.1, freq=0.1, rep=1.1, nblock=3)


def prepare(case, seed):
    d = _dims(case)
    w = {n: t.cpu().numpy() for n, t in _weights(case, seed).items()}
    m = engine.Model(d, stacks=w)
    ids = _ids(case, seed)
    B, n = ids.shape
    st = {"case": case, "ids": ids}
    steps = case.get("steps", 1)
    m.set_rope(*_rope(n + steps + 1, d.head_dim))
    if case.get("f16"):
        m.set_forward_f16(True)
    k = case["kind"]
    if k == "forward":
        rows, T = B, n - 1
        st["d_ids"] = torch.from_numpy(ids[:, :-1].copy()).cuda()
        st["d_tgt"] = torch.from_numpy(ids[:, 1:].copy()).cuda()
        st["logits"] = torch.empty(rows, T, d.vocab, dtype=torch.float32, device="cuda")
        st["nll"] = torch.empty(rows, T, dtype=torch.float32, device="cuda")
        st["stream"] = torch.cuda.Stream()
    elif k == "eval":
        st["token_bytes"] = _token_bytes(seed, d.vocab)
    else:
        st["kv"] = m.kv(B, n + steps + 1, bf16=case.get("kv16", False))
        if k != "prompt":  # the context before the pending id
            for s in range(0, n - 1, 512):
                st["kv"].step_multi(ids[:, s:min(s + 512, n - 1)], want_logits=False)
    st["m"] = m
    torch.cuda.synchronize()
    return st


def run(state):
    case, m = state["case"], state["m"]
    k = case["kind"]
    if k == "forward":
        # on a stream of the caller's, ordered with torch's current one
        s, cur = state["stream"], torch.cuda.current_stream()
        s.wait_stream(cur)
        m.forward_dev(state["d_ids"].data_ptr(), case["B"], case["T"], state["logits"].data_ptr(),
                      state["d_tgt"].data_ptr() if case["nll"] else 0,
                      state["nll"].data_ptr() if case["nll"] else 0, s.cuda_stream)
        cur.wait_stream(s)
        return (state["logits"], state["nll"]) if case["nll"] else (state["logits"],)
    if k == "eval":
        r = m.eval_bpb(state["ids"], state["token_bytes"], batch=case["batch"], want_nll=True)
        return r["nll"], r["row_nats"], r["row_bytes"], r["bpb"]
    kv, ids = state["kv"], state["ids"]
    if k == "prompt":
        kv.len = 0
        npre = case["P"] - 1
        for s in range(0, npre, case["chunk"]):
            kv.step_multi(ids[:, s:min(s + case["chunk"], npre)], want_logits=False)
        lg, nxt = kv.step(ids[:, -1])
        return nxt, lg
    kv.len = case["ctx"]
    if k == "decode":
        return kv.decode_greedy(ids[:, -1], case["steps"], want_logits=True)
    if k == "sample":
        gen, rng = kv.decode_sample(ids[0], case["steps"], seed=12345, **SAMPLING)
        lg, _ = kv.step(gen[-1:])
        return gen, rng, lg
    lg, nxt = kv.step(ids[:, -1])
    return nxt, lg


# ------------------------------------------------------------------ what a call cannot do without

def _matrix_params(case):
    L, D, H, KH, hd, V = SHAPES[case["model"]]
    return L * (2 * H * hd * D + 2 * KH * hd * D + 8 * D * D)


def work(case):
    L, D, H, KH, hd, V = SHAPES[case["model"]]
    B, n = _rows(case)
    layers, head = _matrix_params(case), V * D
    kvb = 2 * KH * hd * L * (2 if case.get("kv16") else 4)  # cache bytes of a position

    def chunk(rows, T, pos0, n_head):  # rows sequences of T positions after pos0, n_head rows of lm_head
        pairs = T * pos0 + T * (T + 1) / 2
        return 2.0 * rows * T * layers + 2.0 * n_head * head + 4.0 * hd * H * L * rows * pairs

    k = case["kind"]
    if k == "forward":
        T = n - 1
        out = B * T * V * 4 + (B * T * 8 if case["nll"] else 0)
        return {"bytes": 2.0 * (layers + head) + B * T * (2.0 * D + 4) + out,
                "flops": chunk(B, T, 0, B * T)}
    if k == "eval":
        T = n - 1
        return {"bytes": 2.0 * (layers + head) + B * T * (2.0 * D + 12) + V * 4,
                "flops": chunk(B, T, 0, B * T)}
    if k == "prompt":
        npre, passes = n - 1, -(-(n - 1) // case["chunk"])
        by = (passes + 1) * 2.0 * layers + 2.0 * head + n * (2.0 * D + kvb) + n * kvb + V * 4
        by += sum(s * kvb for s in range(0, npre, case["chunk"]))  # the cached positions each chunk reads
        return {"bytes": by, "flops": chunk(1, n, 0, 1)}
    steps = case.get("steps", 1) + (1 if k == "sample" else 0)
    by = fl = 0.0
    for s in range(steps):
        length = case["ctx"] + s + 1
        by += 2.0 * (layers + head) + B * (2.0 * D + kvb * (length + 1))
        by += B * V * 4 if k != "sample" or s == steps - 1 else 0
        fl += B * (2.0 * (layers + head) + 4.0 * hd * H * L * length)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # Relative 2-norm, four times what the engine shows against 64 bits. The
    # fp16 pass rounds every operand to 11 bits (logits 4.1e-4, a row's
    # cross-entropy 7e-5); the default one carries ~16 bits of each activation
    # through the MFMA (4.9e-6); a bf16 cache rounds K and V, and another
    # summation order moves some of those roundings by a bf16 ulp (up to
    # 1.3e-4). Ids may differ at near-ties.
    if case.get("f16"):
        return {"rel": 1.6e-3 if case["kind"] == "forward" else 3e-4, "differ": 0.01}
    if case.get("kv16"):
        return {"rel": 5e-4, "differ": 0.01}
    return {"rel": 2e-5, "differ": 0.01}


# ------------------------------------------------------------------ 64 bits

def _norm(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


class _Exact:
    """The model in float64 with a cache, plain torch on the GPU."""

    def __init__(self, case, seed, cap):
        self.s = SHAPES[case["model"]]
        L, D, H, KH, hd, V = self.s
        w = _weights(case, seed)
        rows = {"c_q": H * hd, "c_k": KH * hd, "c_v": KH * hd, "c_proj": D, "c_fc": 4 * D, "c_proj2": D}
        self.w = {n: w[n].view(L, rows[n], -1) for n in LAYER_STACKS}
        self.wte, self.lm = w["wte"].view(V, D), w["lm_head"].view(V, D)
        c, s = _rope(cap, hd)
        self.cos = torch.from_numpy(c).cuda().double()[None, :, None, :]
        self.sin = torch.from_numpy(s).cuda().double()[None, :, None, :]
        self.kv16 = case.get("kv16", False)
        self.k, self.v, self.len = [None] * L, [None] * L, 0

    def _rot(self, x, p0):
        T, h = x.shape[1], x.shape[-1] // 2
        c, s = self.cos[:, p0:p0 + T], self.sin[:, p0:p0 + T]
        a, b = x[..., :h], x[..., h:]
        return torch.cat([a * c + b * s, b * c - a * s], -1)

    def _attend(self, q, k, v, p0):
        """q [B, T, H, hd] at positions p0.., k and v [B, n, KH, hd]."""
        B, T, H, hd = q.shape
        n, rep = k.shape[1], H // k.shape[2]
        hidden = torch.arange(n, device=q.device)[None, :] > (p0 + torch.arange(T, device=q.device))[:, None]
        out = torch.empty_like(q)
        for b in range(B):
            for h in range(H):
                sc = (q[b, :, h] @ k[b, :, h // rep].t().contiguous()) / math.sqrt(hd)
                sc.masked_fill_(hidden, float("-inf"))
                out[b, :, h] = torch.softmax(sc, -1) @ v[b, :, h // rep].contiguous()
        return out.reshape(B, T, H * hd)

    def _attend_one(self, q, k, v):
        B, T, H, hd = q.shape
        rep = H // k.shape[2]
        k = k.repeat_interleave(rep, 2) if rep > 1 else k
        v = v.repeat_interleave(rep, 2) if rep > 1 else v
        p = torch.softmax((k * q).sum(-1) / math.sqrt(hd), 1)
        return (p[..., None] * v).sum(1, keepdim=True).reshape(B, 1, H * hd)

    def hidden(self, ids, keep=True):
        """Final normalised rows [B, T, D] of ids [B, T] at the next positions."""
        L, D, H, KH, hd, V = self.s
        B, T = ids.shape
        p0 = self.len
        x = _norm(self.wte[ids.long()].double())
        for l in range(L):
            W = {n: self.w[n][l].double().t().contiguous() for n in LAYER_STACKS}
            xn = _norm(x)
            q = self._rot((xn @ W["c_q"]).view(B, T, H, hd), p0)
            k = self._rot((xn @ W["c_k"]).view(B, T, KH, hd), p0)
            v = (xn @ W["c_v"]).view(B, T, KH, hd)
            if self.kv16:  # the cache's element type
                k, v = k.to(torch.bfloat16).double(), v.to(torch.bfloat16).double()
            if self.k[l] is not None:
                k, v = torch.cat([self.k[l], k], 1), torch.cat([self.v[l], v], 1)
            if keep:
                self.k[l], self.v[l] = k, v
            ao = self._attend_one(q, k, v) if T == 1 else self._attend(q, k, v, p0)
            x = x + ao @ W["c_proj"]
            h = (_norm(x) @ W["c_fc"]).clamp_(min=0)
            x = x + (h * h) @ W["c_proj2"]
        if keep:
            self.len += T
        return _norm(x)

    def logits(self, h):
        return h @ self.lm.double().t().contiguous()


def _nll(lg, tgt):
    return torch.logsumexp(lg, -1) - lg.gather(-1, tgt.long()[..., None])[..., 0]


@torch.no_grad()
def exact(case, seed):
    k = case["kind"]
    ids = torch.from_numpy(_ids(case, seed)).cuda()
    B, n = ids.shape
    if k == "sample":
        return None  # the draws are the generator's: no value in 64 bits
    ex = _Exact(case, seed, n + case.get("steps", 1) + 1)
    if k in ("forward", "eval"):
        lgs, nlls = [], []
        for b in range(B):  # a row at a time: the fp64 scores are large
            ex.k, ex.v, ex.len = [None] * ex.s[0], [None] * ex.s[0], 0
            lg = ex.logits(ex.hidden(ids[b:b + 1, :-1], keep=False))
            nlls.append(_nll(lg, ids[b:b + 1, 1:]))
            if k == "forward":
                lgs.append(lg)
        nll = torch.cat(nlls)
        if k == "forward":
            return (torch.cat(lgs), nll) if case["nll"] else (torch.cat(lgs),)
        tb = torch.from_numpy(_token_bytes(seed, ex.s[5])).cuda()[ids[:, 1:].long()]
        nats = (nll * (tb > 0)).sum(1)
        by = tb.sum(1)
        bpb = float(nats.sum() / by.sum()) / math.log(2.0)
        return nll.cpu().numpy(), nats.cpu().numpy(), by.cpu().numpy().astype(np.int64), bpb
    if n > 1:
        ex.hidden(ids[:, :-1])
    nxt, out_ids, out_lg = ids[:, -1:], [], []
    for _ in range(case.get("steps", 1)):
        lg = ex.logits(ex.hidden(nxt))[:, 0]
        nxt = lg.argmax(-1, keepdim=True)
        out_ids.append(nxt[:, 0])
        out_lg.append(lg)
    if k == "decode":
        return torch.stack(out_ids).cpu().numpy().astype(np.int32), torch.stack(out_lg).cpu().numpy()
    return out_ids[0].cpu().numpy().astype(np.int32), out_lg[0].cpu().numpy()
