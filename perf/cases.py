"""The workloads that performance work on the library is measured on: what a serving loop calls.

Every case is one call of the public interface (the ctypes mirror of include/g4v.h) on device 0:
verify passes (a tree of two branches, chains, one-row decode) on the synthetic 35-layer stack and
on the Gemma-4-E2B layout, in exact float and with W4A8 products; prompt passes from a short chat
turn to the long-prompt workload; the MTP drafter's chain; the certified head on its own; and the
split-KV attention on device buffers.  Calls return after their work is done, as the interface says.

The library's results are bit-identical to the engine it restates (that is its contract, and every
GPU test holds it to that), so the tolerance of every case is "exact": tokens, counts, hidden
states, logits and attention outputs alike.
"""
import importlib.util
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

V, NL, I, H, HD, NH = 262144, 35, 6144, 1536, 256, 8
WINDOW = 512
GM_MLP = [6144 if l < 15 else 12288 for l in range(35)]
CANDS = 30000  # the most candidates that a row keeps
MOTIF = 64  # the long-prompt workload's prompt: a repeated motif with 5% uniform noise tokens

_G4V = None


def _g4v():
    global _G4V
    if _G4V is None:
        spec = importlib.util.spec_from_file_location("g4v", os.path.join(ROOT, "gemma4-e2b-laptop-cpu_amd", "g4v.py"))
        _G4V = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(_G4V)
    return _G4V


def listed():
    return [
        # the benchmark's step: a 2 x 3 draft tree none of whose drafts are accepted, exact float
        dict(name="verify_tree_2x3_ctx2048", kind="verify", gemma=False, ctx=2048, na=3, nb=3, int8=False, accept=False,
             nsplit=8),
        # a decode round of the long-prompt workload: a chain of 3 drafts that the model accepts
        dict(name="verify_chain3_accept_ctx6841", kind="verify", gemma=False, ctx=6841, na=3, nb=0, int8=False,
             accept=True, nsplit=8),
        # plain decode, one row a pass, on the checkpoint's layout
        dict(name="gemma_decode1_ctx2048", kind="verify", gemma=True, ctx=2048, na=0, nb=0, int8=False, accept=False,
             nsplit=6),
        # a speculative round in the server's mode (W4A8 products) on the checkpoint's layout
        dict(name="gemma_chain3_w4a8_ctx2048", kind="verify", gemma=True, ctx=2048, na=3, nb=0, int8=True, accept=False,
             nsplit=6),
        # the longest chain a prompt lookup drafts (8 rows), early in a conversation, exact float
        dict(name="gemma_chain7_ctx1003", kind="verify", gemma=True, ctx=1003, na=7, nb=0, int8=False, accept=False,
             nsplit=6),
        # the long-prompt workload's prompt
        dict(name="prefill_motif_6841", kind="prefill", gemma=False, n=6841, int8=True, pfb=32, nsplit=8),
        # a short chat turn
        dict(name="prefill_40", kind="prefill", gemma=False, n=40, int8=True, pfb=32, nsplit=8),
        # a ragged prompt of ordinary length without W4A8 (the engine's default arithmetic)
        dict(name="prefill_exact_333", kind="prefill", gemma=False, n=333, int8=False, pfb=32, nsplit=8),
        # a ragged document prompt on the checkpoint's layout
        dict(name="gemma_prefill_1531", kind="prefill", gemma=True, n=1531, int8=True, pfb=32, nsplit=6),
        # the drafter's chain of a speculative round
        dict(name="draft_mtp3_ctx2048", kind="draft", ctx=2048, k=3, nsplit=6),
        # the head alone: two rows the screen prunes and two that fall back to the full head
        dict(name="head_4rows", kind="head", aligned=2, random=2),
        # attention alone, as a loop with its own caches calls it: the smallest call here
        dict(name="attn_4rows_2048", kind="attn", npos=2048, M=4, window=False, nsplit=8),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["verify", "verify", "verify", "prefill", "prefill", "draft", "head", "attn"])
    if kind == "verify":
        gemma = rng.random() < 0.5
        form = rng.choice(["decode", "chain", "chain", "tree"])
        if gemma and form == "tree":  # that layout takes chains and one sibling row
            form = "chain"
        na, nb = {"decode": (0, 0), "chain": (rng.randint(1, 7), 0), "tree": (rng.randint(1, 3), rng.randint(1, 4))}[form]
        return dict(kind=kind, gemma=gemma, ctx=_log(rng, 24, 4000 if gemma else 7900), na=na, nb=nb,
                    int8=rng.random() < 0.4, accept=rng.random() < 0.4, nsplit=rng.choice([6, 8]))
    if kind == "prefill":
        gemma = rng.random() < 0.5
        return dict(kind=kind, gemma=gemma, n=_log(rng, 9, 2500 if gemma else 5000), int8=rng.random() < 0.7,
                    pfb=rng.choice([32, 32, 16]), nsplit=rng.choice([6, 8]))
    if kind == "draft":
        return dict(kind=kind, ctx=_log(rng, 16, 7900), k=rng.randint(1, 4), nsplit=rng.choice([6, 8]))
    if kind == "head":
        n = rng.randint(1, 4)
        a = rng.randint(0, n)
        return dict(kind=kind, aligned=a, random=n - a)
    return dict(kind=kind, npos=_log(rng, 48, 4096), M=rng.randint(1, 8), window=rng.random() < 0.5,
                nsplit=rng.choice([4, 6, 8, 16]))


def _prompt(n, seed):
    rng = np.random.default_rng(seed)
    toks = np.resize(rng.integers(0, V, MOTIF), n).astype(np.int32)
    noise = rng.random(n) < 0.05
    toks[noise] = rng.integers(0, V, int(noise.sum()))
    return toks


def _model(case, seed, ctxcap):
    dev = _g4v().Device(0)
    if case.get("gemma"):
        dev.model_synth_gemma(seed, V, np.array(GM_MLP, np.int32), ctxcap)
    else:
        dev.model_synth(seed, V, NL, I, ctxcap)
    return dev


def _attn_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    npos, M = case["npos"], case["M"]
    K, Vv = (torch.randn(npos, HD, generator=g, device="cuda").bfloat16() for _ in range(2))
    q = (torch.randn(M, NH * HD, generator=g, device="cuda") / 16).float()  # normed, scaled heads
    pos = np.arange(npos - M, npos, dtype=np.int32)
    lo = np.maximum(0, pos - (WINDOW - 1)).astype(np.int32) if case["window"] else np.zeros(M, np.int32)
    return K, Vv, q, pos, lo


def _head_inputs(case, seed):
    """an embedding of the checkpoint's shape; rows aligned with an entry of it at varied strengths
    (a confident model) and rows that are not"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    E = (torch.randn(V, H, generator=g, device="cuda") * 0.02).bfloat16()
    rows = []
    for m in range(case["aligned"]):
        at = int(torch.randint(0, V, (1,), generator=g, device="cuda"))
        rows.append(E[at].float() * (16.0 + 8.0 * m) + torch.randn(H, generator=g, device="cuda"))
    for _ in range(case["random"]):
        rows.append(torch.randn(H, generator=g, device="cuda"))
    return E, torch.stack(rows).bfloat16().float()


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed + 1)
    if kind == "verify":
        M = 1 + case["na"] + case["nb"]
        dev = _model(case, seed, 4096 if case["ctx"] + M <= 4096 else 8192)
        dev.fake_ctx(case["ctx"], seed)
        if case["int8"]:
            dev.set_decode_int8(True)
        toks = rng.integers(0, V, M).astype(np.int32)
        if case["accept"]:  # the random-init stack's greedy token repeats the row's own token
            toks[1:1 + case["na"]] = toks[0]
        return dict(case=case, dev=dev, toks=toks)
    if kind == "prefill":
        dev = _model(case, seed, 4096 if case["n"] <= 4000 else 8192)
        dev.set_prefill_int8(case["int8"])
        return dict(case=case, dev=dev, toks=_prompt(case["n"], seed))
    if kind == "draft":
        dev = _model(case, seed, 4096 if case["ctx"] <= 4000 else 8192)
        dev.fake_ctx(case["ctx"], seed)
        dev.drafter_synth(seed + 1)
        return dict(case=case, dev=dev, tok=int(rng.integers(0, V)), h=rng.standard_normal(H).astype(np.float32))
    if kind == "head":
        dev = _g4v().Device(0)
        E, h = _head_inputs(case, seed)
        dev.head_build(E.view(torch.int16).cpu().numpy().view(np.uint16), V)
        return dict(case=case, dev=dev, h=h.cpu().numpy())
    dev = _g4v().Device(0)
    K, Vv, q, pos, lo = _attn_inputs(case, seed)
    out = torch.empty_like(q)
    torch.cuda.synchronize()  # the inputs are there before the library's own stream reads them
    return dict(case=case, dev=dev, K=K, V=Vv, q=q, pos=pos, lo=lo, none=(np.ones_like(pos), np.zeros_like(pos)), out=out)


def run(state):
    case, dev = state["case"], state["dev"]
    kind = case["kind"]
    if kind == "verify":
        r, hidden = dev.verify(state["toks"], case["na"], case["nb"], case["ctx"], case["nsplit"], hidden=True)
        commit = np.array(r.commit[:r.ncommit] + [-1] * (8 - r.ncommit))
        return dict(nacc=r.nacc, branch=r.branch, ncommit=r.ncommit, commit=commit, G=np.array(r.G[:]),
                    fallback=np.array(r.fallback[:]), nsurv=np.array(r.nsurv[:]), hidden=hidden)
    if kind == "prefill":
        g0, hidden = dev.prefill(state["toks"], 0, case["pfb"], case["nsplit"], hidden=True)
        return dict(token=g0, hidden=hidden)
    if kind == "draft":
        d, sec, gap, hidden = dev.draft_mtp(state["tok"], state["h"], case["ctx"] - 1, case["k"], case["nsplit"])
        return dict(drafts=d, second=sec, gap=gap, hidden=hidden)
    if kind == "head":
        G, ns, fb = dev.head_argmax(state["h"])
        out = dict(G=G, nsurv=ns, fallback=fb, candidates=np.full(CANDS, -1, np.int32), logits=np.zeros(CANDS, np.float32))
        if not fb[0]:  # the candidates of the first row, with their logits (a row of too many has none)
            idx, val, n = dev.head_survivors(0)
            out["candidates"][:n], out["logits"][:n] = idx, val
        return out
    pos, lo = state["pos"], state["lo"]
    dev.attn_noalloc(state["K"].data_ptr(), state["V"].data_ptr(), case["npos"], state["q"].data_ptr(), case["M"], pos, lo,
                     *state["none"], int(lo.min()), int(pos[-1]), case["nsplit"], state["out"].data_ptr())
    return state["out"]


def _q4(n, k):
    return n * k // 2 + n * k // 16


def _layers(gemma):
    """(matrix bytes, parameters, attention head dim, sliding window) of each layer"""
    out = []
    for l in range(NL):
        hd = 512 if gemma and l % 5 == 4 else 256
        mlp = GM_MLP[l] if gemma else I
        shapes = [(NH * hd, H), (H, NH * hd), (mlp, H), (mlp, H), (H, mlp)]
        if not gemma or l < 15:
            shapes += [(hd, H)] * 2
        if gemma:
            shapes += [(256, H), (H, 256), (256, H)]  # the per-layer-input gate, projection and share of the model's
        out.append((sum(_q4(*s) for s in shapes), sum(n * k for n, k in shapes), hd, l % 5 != 4))
    return out


SCREEN = _q4(V, H) + 4 * V


def _keys(first, n, sliding):
    """(keys read at least once, keys scored) by rows at positions first .. first + n - 1"""
    if not sliding:
        return first + n, n * first + n * (n + 1) // 2
    p = np.arange(first, first + n, dtype=np.int64)
    return min(first + n, WINDOW - 1 + n), int(np.minimum(p + 1, WINDOW).sum())


def work(case):
    kind = case["kind"]
    if kind in ("verify", "prefill"):
        first, n = (case["ctx"], 1 + case["na"] + case["nb"]) if kind == "verify" else (0, case["n"])
        nbytes, flops = SCREEN, 2 * V * H  # the head of one row
        for mb, params, hd, sliding in _layers(case["gemma"]):
            read, scored = _keys(first, n, sliding)
            nbytes += mb + read * hd * 2 * 2
            flops += 2 * params * n + 2 * 2 * scored * NH * hd
        if kind == "prefill":
            nbytes += n * H * 2
        return dict(bytes=nbytes, flops=flops)
    if kind == "draft":
        # bf16: the projections, four layers (4 heads of 256, FFN 2048), centroids, 32 x 128 candidates
        params = 2 * H * 256 + H * 256 + 4 * (2 * 1024 * 256 + 3 * 2048 * 256) + V // 128 * 256 + 4096 * 256
        keys = 3 * min(case["ctx"], WINDOW) + case["ctx"]
        return dict(bytes=case["k"] * (2 * params + keys * HD * 4), flops=case["k"] * (2 * params + 16 * keys * HD))
    if kind == "head":
        full = 44 * V * H // 32 if case["random"] else 0  # the 11-bit exponent-coded rows, once for every row
        return dict(bytes=SCREEN + full, flops=2 * V * H * (case["aligned"] + 2 * case["random"]))
    read, scored = _keys(case["npos"] - case["M"], case["M"], case["window"])
    return dict(bytes=read * HD * 4 + case["M"] * NH * HD * 8, flops=4 * scored * NH * HD)


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Attention in 64 bits.  The whole passes have none: they round to bf16 after every block by
    definition, and what a pass gives follows those roundings through every layer; the head's
    outputs are whole numbers and the logits rounded to bf16 of a set that its screen chooses."""
    if case["kind"] != "attn":
        return None
    K, Vv, q, pos, lo = _attn_inputs(case, seed)
    at = torch.arange(case["npos"], device="cuda")
    pos, lo = (torch.from_numpy(x).cuda() for x in (pos, lo))
    s = q.double().view(case["M"], NH, HD) @ K.double().T
    s = s.masked_fill(((at > pos[:, None]) | (at < lo[:, None]))[:, None], -math.inf)
    return (torch.softmax(s, -1) @ Vv.double()).reshape(case["M"], NH * HD)
