"""The sampler calls a serving program makes, with the inputs it makes them on.

A program that serves a model calls the C ABI of include/ferro_sampler.h once per generated token (or per speculative
window), from C++, with device pointers it already holds. The cases here make the same calls through the package's
ctypes binding of that ABI. Logit, history and parameter distributions are those of ferro_amd/workloads.py; vocabulary
sizes are the 65536 and 262144 used throughout this repository, and one that is no multiple of anything.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import ferro_amd as F
from ferro_amd._lib import check, lib

# ferro::SamplerParams' defaults: what a client gets that sets nothing (near-greedy, the whole history penalised)
DEFAULTS = dict(T=0.05, k=50, p=1.0, min_p=0.0, rep=1.05, freq=0.0, pres=0.0, last_n=-1, softcap=0.0)


def _case(name, call, B, V, H, logits, **kw):
    """call: the entry point. B rows (verify, draft: streams) of V logits; H history ids per row, on the average where
    ragged. mixed: every row has parameters of its own."""
    c = dict(name=name, call=call, B=B, V=V, H=H, logits=logits, ragged=False, mixed=False, M=1, kcap=0)
    c.update(DEFAULTS)
    c.update(kw)
    return c


def listed():
    return [
        # one interactive session: a single row per token, nucleus sampling over a short penalty window
        _case("chat_row", "sample", 1, 65536, 64, "spikes", T=0.7, k=40, p=0.95, rep=1.1),
        # a small greedy batch with frequency / presence penalties (deterministic structured output)
        _case("greedy_counts", "sample", 8, 65536, 256, "normal", T=0.0, rep=1.0, freq=0.5, pres=0.3),
        # the serving batch: 64 sessions on the large vocabulary, top-k 64 / top-p
        _case("serving", "sample", 64, 262144, 512, "mixture", T=0.8, k=64, p=0.95),
        # speculative decoding, greedy: 16 streams verify 16 drafts and a bonus row each
        _case("verify_greedy", "verify", 16, 65536, 64, "normal", T=0.0, rep=1.0, M=17),
        # speculative decoding on the server's default parameters: sampled rows, the history and the drafts penalised
        _case("verify_default", "verify", 8, 262144, 1024, "mixture", M=5, ragged=True),
        # a large batch of clients that each set their own parameters
        _case("mixed_clients", "sample", 256, 262144, 1024, "mixture", mixed=True),
        # top-p alone (top_k = 0: every token is a candidate), the usual setting of OpenAI-style clients
        _case("nucleus", "sample", 64, 262144, 512, "mixture", T=0.8, k=0, p=0.95),
        # plain sampling at temperature 1 with no cut (rollouts, evaluation), on high-entropy rows
        _case("rollout_flat", "sample", 32, 65536, 0, "normal", T=1.0, k=0, rep=1.0),
        # long conversations on the default parameters with the model's final softcap, the decode step in one launch
        _case("long_context", "decode", 8, 262144, 16384, "mixture", softcap=30.0, ragged=True),
        # the decode step of a medium batch with ragged histories
        _case("decode_step", "decode", 32, 65536, 700, "spikes", T=0.7, k=40, p=0.95, rep=1.1, ragged=True),
        # wider top-k with frequency / presence penalties, the top 20 candidates' probabilities returned, odd vocabulary
        _case("logprobs_wide_k", "sample", 24, 100003, 400, "mixture", T=0.9, k=200, p=0.9, rep=1.0, freq=0.2, pres=0.1,
              kcap=20, ragged=True),
        # prompt-lookup drafting before a verification window: 64 streams' histories searched
        _case("draft_lookup", "draft", 64, 65536, 8192, "none", ragged=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the same kinds: every size over its range, odd ones among them."""
    base = dict(rng.choice(listed()))
    del base["name"]
    V = rng.choice([65536, 262144, rng.randint(32000, 262144), rng.randint(32000, 262144)])
    # logits a drawn case may read: no more than the listed case of its kind
    cap = (1 << 26) if base["mixed"] else (1 << 21) if base["logits"] == "normal" and base["k"] == 0 else 1 << 24
    if base["call"] == "draft":
        base.update(B=_log_int(rng, 1, 128), V=V, H=_log_int(rng, 64, 16384))
        return base
    if base["call"] == "verify":
        base["M"] = rng.randint(2, 17)
    rows = max(1, min(256, cap // V))
    base.update(V=V, B=max(1, _log_int(rng, 1, rows) // base["M"]))
    if base["H"]:
        base["H"] = _log_int(rng, 16, 16384 if base["B"] <= 16 else 2048)
    if base["T"] > 0 and not base["mixed"]:
        base["T"] = round(rng.uniform(0.05, 1.3), 2)
        if base["k"]:
            base["k"] = _log_int(rng, 65, 1024) if base["k"] > 64 else rng.randint(10, 64)
            base["p"] = rng.choice([1.0, round(rng.uniform(0.8, 1.0), 3)])
            base["min_p"] = rng.choice([0.0, 0.0, 0.05])
    return base


# ------------------------------------------------------------------------------------------------ inputs
def _logits(kind, R, V, ld, g):
    x = torch.empty((R, ld), dtype=torch.float32, device="cuda")
    randn = functools.partial(torch.randn, dtype=torch.float32, device="cuda", generator=g)
    if kind == "mixture":              # 90% N(0, 1.5), 10% Student-t(3) * 4
        z = randn(R, ld)
        chi = randn(R, ld).square_().add_(randn(R, ld).square_()).add_(randn(R, ld).square_())
        t = 4.0 * z * torch.rsqrt(chi / 3.0)
        pick = torch.rand((R, ld), device="cuda", generator=g) < 0.1
        torch.where(pick, t, 1.5 * z, out=x)
    else:
        x.copy_(2.0 * randn(R, ld))
        if kind == "spikes":           # 8 tokens of each row stand out by 12
            at = torch.randint(0, V, (R, 8), device="cuda", generator=g)
            x.scatter_add_(1, at, torch.full((R, 8), 12.0, device="cuda"))
    return x


def _histories(case, rs):
    """CSR histories of Zipf(1.1) ids; ragged: lengths from a quarter of H to 7/4 of it."""
    S, V, H = case["B"], case["V"], case["H"]
    n = np.full(S, H)
    if case["ragged"] and S > 1:       # the same lengths for every seed, on other rows
        n = rs.permutation(np.linspace(H // 4, 2 * H - H // 4, S).astype(np.int64))
    off = np.zeros(S + 1, np.int64)
    off[1:] = np.cumsum(n)
    cdf = np.cumsum(np.arange(1, V + 1, dtype=np.float64) ** -1.1)
    ids = np.searchsorted(cdf, rs.random_sample(int(off[-1])) * cdf[-1]).clip(0, V - 1).astype(np.int32)
    if case["call"] == "draft":        # half of the streams repeat an earlier passage at their end, as edited text does
        for s in range(0, S, 2):
            if n[s] >= 16:
                a = off[s] + rs.randint(0, n[s] - 12)
                ids[off[s + 1] - 4:off[s + 1]] = ids[a:a + 4]
    return ids, off


def _params(case, rs):
    B = case["B"]
    p = np.zeros(B, F.PARAMS_DTYPE)
    for field, key in (("temperature", "T"), ("top_k", "k"), ("top_p", "p"), ("min_p", "min_p"),
                       ("repetition_penalty", "rep"), ("frequency_penalty", "freq"), ("presence_penalty", "pres"),
                       ("repeat_last_n", "last_n"), ("softcap", "softcap")):
        p[field] = case[key]
    if case["mixed"]:
        T = rs.uniform(0.3, 1.5, B)
        T[rs.random_sample(B) < 0.05] = 0.0
        p["temperature"] = T
        p["top_k"] = np.floor(np.exp(rs.uniform(0.0, math.log(2048.0), B))).astype(np.int32).clip(1, 2048)
        p["top_p"] = rs.uniform(0.8, 1.0, B)
        p["repetition_penalty"] = rs.uniform(1.0, 1.3, B)
        p["frequency_penalty"] = rs.uniform(0.0, 1.0, B)
        p["presence_penalty"] = rs.uniform(0.0, 1.0, B)
    return p


def _inputs(case, seed):
    """Everything made from the seed: logits, histories, parameters, draws and (verify) the fed tokens."""
    rs = np.random.RandomState(seed % (1 << 32))
    g = torch.Generator("cuda").manual_seed(seed)
    B, V, M = case["B"], case["V"], case["M"]
    d = {"ld": -(-V // 128) * 128}     # an lm_head writes its rows padded to a multiple of 128
    if case["H"]:
        ids, off = _histories(case, rs)
        d["hist_n"] = int(off[-1])
        d["hist"], d["off"] = torch.from_numpy(ids).cuda(), torch.from_numpy(off).cuda()
    if case["call"] == "draft":
        d["kmax"] = torch.full((B,), 16, dtype=torch.int32, device="cuda")
        return d
    d["x"] = _logits(case["logits"], B * M, V, d["ld"], g)
    d["hp"] = _params(case, rs)
    d["p"] = torch.from_numpy(d["hp"].view(np.uint8).copy()).cuda()
    d["u"] = torch.from_numpy(rs.random_sample(B * M)).cuda()
    if case["call"] == "verify":       # a draft is the row's largest logit four times out of five
        best = d["x"][:, :V].argmax(1).cpu().numpy().reshape(B, M)
        rows = rs.randint(0, V, (B, M))
        rows[:, 1:] = np.where(rs.random_sample((B, M - 1)) < 0.8, best[:, :-1], rows[:, 1:])
        d["rows"] = torch.from_numpy(rows.reshape(-1).astype(np.int32)).cuda()
        d["row_off"] = torch.arange(0, B * M + 1, M, dtype=torch.int64, device="cuda")
    if case["call"] == "decode":
        d["seeds"] = rs.randint(1, 1 << 31, B).astype(np.uint64)
    return d


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    d = _inputs(case, seed)
    L, ctx = lib(), F.Context.default()
    B, V, M = case["B"], case["V"], case["M"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    i32 = functools.partial(torch.zeros, dtype=torch.int32, device="cuda")
    hist, off = d.get("hist"), d.get("off")
    keep = [d, ctx]
    if case["call"] == "draft":
        out = {"draft": i32((B, 16)), "n": i32(B)}
        fn, args = L.fs_lookup_draft, (ctx.h, B, _ptr(hist), _ptr(off), _ptr(d["kmax"]), None, -1, _ptr(out["draft"]), 16,
                                       _ptr(out["n"]), stream)
        return {"fn": functools.partial(fn, *args), "out": out, "keep": keep}
    rows = (ctx.h, _ptr(d["x"]), d["ld"])
    hp = d["hp"].ctypes.data_as(ctypes.c_void_p)
    if case["call"] == "sample":
        out = {"tok": i32(B), "keep": i32(B)}
        if case["kcap"]:
            out["ids"] = i32((B, case["kcap"]))
            out["probs"] = torch.zeros((B, case["kcap"]), dtype=torch.float64, device="cuda")
        fn, args = L.fs_sample_batch_hp, rows + (
            B, V, _ptr(hist), _ptr(off), _ptr(d["p"]), hp, _ptr(d["u"]), _ptr(out["tok"]), case["kcap"],
            _ptr(out.get("ids")), _ptr(out.get("probs")), _ptr(out["keep"]), stream)
    elif case["call"] == "verify":
        out = {"tok": i32(B * M), "accepted": i32(B)}
        fn, args = L.fs_verify_hp, rows + (
            B, B * M, V, _ptr(d["rows"]), _ptr(d["row_off"]), _ptr(hist), _ptr(off), _ptr(d["p"]), hp, _ptr(d["u"]), -1,
            _ptr(out["tok"]), _ptr(out["accepted"]), stream)
    else:
        rng = F.DeviceRng(d["seeds"])
        keep.append(rng)
        cap = d["hist_n"] + B
        out = {"tok": i32(B), "keep": i32(B), "hist": i32(cap),
               "off": torch.zeros(B + 1, dtype=torch.int64, device="cuda")}
        fn, args = L.fs_decode_step_hp, (ctx.h, rng.h) + rows[1:] + (
            B, V, _ptr(hist), _ptr(off), _ptr(d["p"]), hp, _ptr(out["tok"]), _ptr(out["keep"]), _ptr(out["hist"]),
            _ptr(out["off"]), cap, stream)
    return {"fn": functools.partial(fn, *args), "out": out, "keep": keep}


def run(state):
    check(state["fn"](), "the sampling call")
    return state["out"]


# ------------------------------------------------------------------------------------------------ what is compared
def work(case):
    R, V, H = case["B"] * case["M"], case["V"], case["B"] * case["H"]    # H: ids in all
    if case["call"] == "draft":
        return {"bytes": 4 * H + case["B"] * 17 * 4, "flops": H}
    out = R * 8 + case["kcap"] * R * 12
    if case["call"] == "decode":
        out += 4 * H                   # the histories are written once more, a token longer
    return {"bytes": 4 * R * V + 4 * H + out, "flops": R * V * (1 if case["softcap"] == 0 else 20)}


def tolerance(case):
    # Token ids, kept counts, candidate ids, accepted lengths and histories are whole numbers: equal. The probabilities
    # are 64-bit exponentials and sums: 3e-16 off exact() as measured, up to ten times that where a low temperature
    # makes the exponents large.
    return {"rel": 1e-14} if case["kcap"] else "exact"


def exact(case, seed):
    """The candidates' probabilities in 64 bits: penalties over the window, the k largest logits (the lower id first
    among equal ones), softmax at the temperature over the candidates."""
    if not case["kcap"]:
        return None
    d = _inputs(case, seed)
    B, V, kcap = case["B"], case["V"], case["kcap"]
    probs = torch.zeros((B, kcap), dtype=torch.float64, device="cuda")
    for b in range(B):
        x = d["x"][b, :V].double()
        if case["H"]:
            h = d["hist"][int(d["off"][b]):int(d["off"][b + 1])].long()
            n = torch.bincount(h, minlength=V).double()
            rep = float(np.float32(case["rep"]))
            x = torch.where(n > 0, torch.where(x > 0, x / rep, x * rep), x)
            x = x - n * float(np.float32(case["freq"])) - (n > 0).double() * float(np.float32(case["pres"]))
        k = case["k"] if 0 < case["k"] < V else V
        top = torch.sort(x, descending=True, stable=True).values[:k]
        pr = torch.softmax(top / float(np.float32(case["T"])), 0)
        probs[b, :min(k, kcap)] = pr[:kcap]
    return {"probs": probs}
