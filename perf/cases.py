"""The work that this library is asked to do, through its public entry points: what a serving program calls per layer
and step, at the sizes that it calls it with.

Five families, each with its range (see draw()):

- decode: DecodeLayer.step over the paged FP8 caches, one new token per sequence. Batches of 1 to 64 sequences of 500 to
  1M tokens, of one length or ragged; 16, 32, 64 or 128 query heads (a tensor-parallel shard, or all of them).
- pooled: GLM's decode step (kpool 4) with the pool-key write in it, PooledDecodeLayer.step(write=...).
- chunk: a prefill chunk, dsa_long_select.select and then dsa_decode.attend_tokens, with FP8 or bf16 indexer queries,
  from the first chunk of a short prompt to the last one of a long prompt.
- pooled_chunk: GLM's prefill chunk, dsa_long_select.select over bf16 pool keys and then dsa_long.attend_pooled.
- store: the quantise-on-write of new rows into the two paged caches before the layer.

Inputs are the seeded synthetic ones of trnrt_amd.workloads: N(0, 1) keys, latent rows and queries, quantised per token.
"""

from __future__ import annotations

import math
import random

import torch

from trnrt_amd import workloads as W
from trnrt_amd.kernels import dsa_cache, dsa_decode, dsa_layer, dsa_long_select
from trnrt_amd.models import dsa_long

PAGE = 64
KEEP = 2048  # tokens selected per query (512 pools of 4 in the pooled form)
KP = 4
DEV = "cuda"


def listed() -> list[dict]:
    return [
        # one sequence of a short conversation on a tensor-parallel shard: the smallest call, all latency
        dict(name="decode-1x4k-h16", family="decode", B=1, L=4096, low=4096, H=16, Hi=16),
        # the headline step: a small batch at 32K, all rows in one launch
        dict(name="decode-8x32k", family="decode", B=8, L=32768, low=32768, H=64, Hi=64),
        # a full serving batch of conversations of all lengths, several rows to each part of the GPU
        dict(name="decode-48-ragged", family="decode", B=48, L=32768, low=500, H=64, Hi=64),
        # an odd batch with all 128 query heads on one GPU (data-parallel attention), prompts of up to 12,345 tokens
        dict(name="decode-13-h128", family="decode", B=13, L=12345, low=2000, H=128, Hi=64),
        # long documents of different lengths
        dict(name="decode-12x8k-128k", family="decode", B=12, L=131072, low=8192, H=64, Hi=64),
        # the longest context: four sequences of 1M tokens
        dict(name="decode-4x1m", family="decode", B=4, L=1048576, low=1048576, H=64, Hi=64),
        # GLM's step at 32K: pool-key write, pooled indexer, selection and attention
        dict(name="pooled-8x32k", family="pooled", B=8, L=32768, low=32768, H=64, Hi=32),
        # the same step for a full, ragged serving batch
        dict(name="pooled-30-ragged", family="pooled", B=30, L=32000, low=700, H=64, Hi=32),
        # a late chunk of a long prompt with FP8 indexer queries: the largest call
        dict(name="chunk-2048-64k-fp8", family="chunk", N=2048, cached=65536, H=64, Hi=64, q_fp8=True),
        # the ragged last chunk of an ordinary prompt, bf16 indexer queries
        dict(name="chunk-1001-6k-bf16", family="chunk", N=1001, cached=6000, H=64, Hi=64, q_fp8=False),
        # GLM's late chunk of a long prompt
        dict(name="glm-chunk-2048-64k", family="pooled_chunk", N=2048, cached=65536, H=64, Hi=32),
        # a chunk's new rows written into the latent and the indexer-key caches
        dict(name="store-2048", family="store", T=2048, slots=70016, x_fp32=False),
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    """A whole number between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    """One more case of the listed ones' ranges; none costs more than the largest of its family."""
    family = rng.choice(["decode", "decode", "decode", "pooled", "chunk", "chunk", "pooled_chunk", "store"])
    if family == "decode":
        B = _log(rng, 1, 64)
        L = _log(rng, 1000, min(1 << 20, (4 << 20) / B))
        low = L if rng.random() < 0.3 else max(1, int(L * rng.uniform(0.05, 0.9)))
        return dict(family=family, B=B, L=L, low=low, H=rng.choice([16, 32, 64, 64, 128]), Hi=rng.choice([16, 32, 64, 64]))
    if family == "pooled":
        B = _log(rng, 1, 32)
        L = _log(rng, 1000, min(131072, (1 << 20) / B))
        low = L if rng.random() < 0.3 else max(1, int(L * rng.uniform(0.05, 0.9)))
        return dict(family=family, B=B, L=L, low=low, H=rng.choice([32, 64, 64]), Hi=32)
    if family == "store":
        return dict(family=family, T=_log(rng, 1, 8192), slots=64 * rng.randint(128, 2048), x_fp32=rng.random() < 0.3)
    N = _log(rng, 64, 2048)
    cached = 0 if rng.random() < 0.15 else _log(rng, 100, 65536)
    if family == "chunk":
        return dict(family=family, N=N, cached=cached, H=rng.choice([16, 64, 64, 128]) if N <= 1024 else 64,
                    Hi=rng.choice([32, 64, 64]), q_fp8=rng.random() < 0.5)
    return dict(family=family, N=N, cached=cached, H=64, Hi=32)


# -- what a program has in hand before the call -----------------------------------------------------------------


def _lengths(case: dict, seed: int) -> list[int]:
    """The batch's lengths: U[low, L], one of them the longest (so that the shapes follow from the case alone)."""
    g = torch.Generator().manual_seed(seed)
    n = [int(x) for x in torch.randint(case["low"], case["L"] + 1, (case["B"],), generator=g)]
    n[seed % case["B"]] = case["L"]
    return n


def _prepare_decode(case: dict, seed: int) -> dict:
    lengths = _lengths(case, seed)
    cfg = W.Config("case", B=case["B"], L=case["L"], H=case["H"], Hi=case["Hi"], keep=KEEP, page_size=PAGE)
    inp = W.make_inputs(cfg, seed=seed, device=DEV, lengths=lengths)
    layer = dsa_layer.DecodeLayer(case["B"], case["Hi"], case["H"], inp.max_pages, PAGE, inp.num_pages, keep=KEEP,
                                  scale=cfg.scale, device=DEV)
    return dict(case=case, inp=inp, layer=layer)


def _prepare_pooled(case: dict, seed: int) -> dict:
    B, L, H, Hi = case["B"], case["L"], case["H"], case["Hi"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    npg = math.ceil(L / PAGE)
    slots = (1 + B * npg) * PAGE
    rows, rows_scale = W.quantize_rows(torch.randn(slots, 256, generator=g, device=DEV))
    kv = torch.empty(slots, 512, dtype=W.FP8, device=DEV)
    kv_scale = torch.empty(slots, dtype=torch.float32, device=DEV)
    for s in range(0, slots, 262144):
        n = min(262144, slots - s)
        kv[s:s + n], kv_scale[s:s + n] = W.quantize_rows(torch.randn(n, 512, generator=g, device=DEV))
    table = (torch.randperm(B * npg, generator=g, device=DEV) + 1).view(B, npg).to(torch.int32)
    ape = torch.randn(KP, 128, generator=g, device=DEV) * 0.5
    q_idx = torch.randn(B, Hi, 128, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(B, Hi, generator=g, device=DEV) * 0.25 * 128 ** -0.5
    q = torch.randn(B, H, 512, generator=g, device=DEV).to(torch.bfloat16)
    pool_key = torch.zeros(slots, 128 // KP, dtype=torch.bfloat16, device=DEV)
    every = torch.arange(L, device=DEV)
    for b in range(B):  # the context's pool keys, as the steps before this one wrote them
        dsa_cache.write_pool_keys(pool_key, rows, every, table[b], dsa_cache.slots_of(every, table[b], PAGE), ape, PAGE,
                                  KP, rows_scale=rows_scale)
    positions = torch.tensor([n - 1 for n in _lengths(case, seed)], dtype=torch.int32, device=DEV)
    npool = torch.div(positions + 1, KP, rounding_mode="floor").to(torch.int32)
    layer = dsa_layer.PooledDecodeLayer(B, Hi, H, 512, npg, PAGE, slots // PAGE, KP, KEEP // KP, 256 ** -0.5, device=DEV)
    return dict(case=case, layer=layer, rows=rows, rows_scale=rows_scale, kv=kv, kv_scale=kv_scale, table=table, ape=ape,
                q_idx=q_idx, w=w, q=q, pool_key=pool_key, positions=positions, npool=npool,
                slot_mapping=dsa_cache.slots_of(positions, table, PAGE))


def _prepare_chunk(case: dict, seed: int) -> dict:
    cfg = W.PrefillConfig("case", cached=case["cached"], chunk=case["N"], Hi=case["Hi"], keep=KEEP, q_fp8=case["q_fp8"],
                          H=case["H"], page_size=PAGE)
    inp = W.make_prefill_inputs(cfg, seed=seed, device=DEV, attention=True)
    return dict(case=case, inp=inp, tables=inp.table.expand(case["N"], -1).contiguous())


def _prepare_pooled_chunk(case: dict, seed: int) -> dict:
    cfg = W.PooledPrefillConfig("case", cached=case["cached"], chunk=case["N"], Hi=case["Hi"], H=case["H"], kp=KP,
                                topk=KEEP, page_size=PAGE)
    return dict(case=case, inp=W.make_pooled_prefill_inputs(cfg, seed=seed, device=DEV))


def _prepare_store(case: dict, seed: int) -> dict:
    T, slots = case["T"], case["slots"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = torch.float32 if case["x_fp32"] else torch.bfloat16
    at = torch.randperm(slots // PAGE - 1, generator=g, device=DEV)[:math.ceil(T / PAGE)] + 1  # whole pages, any order
    slot_mapping = (at.view(-1, 1) * PAGE + torch.arange(PAGE, device=DEV)).view(-1)[:T].contiguous()
    st = dict(case=case, slot_mapping=slot_mapping)
    for name, width in (("latent", 576), ("key", 128)):
        st[name] = torch.randn(T, width, generator=g, device=DEV).to(dt)
        st[name + "_cache"] = torch.zeros(slots, width, dtype=W.FP8, device=DEV)
        st[name + "_scale"] = torch.ones(slots, dtype=torch.float32, device=DEV)
    return st


def prepare(case: dict, seed: int) -> dict:
    return globals()["_prepare_" + case["family"]](case, seed)


# -- one pass -----------------------------------------------------------------------------------------------------


def _run_decode(s: dict) -> dict:
    i = s["inp"]
    out, lse = s["layer"].step(i.q_idx, i.w_k, i.k_cache, i.k_scale, i.q, i.kv_cache, i.kv_scale, i.table, i.ctx_len)
    return dict(out=out, lse=lse)


def _run_pooled(s: dict) -> dict:
    out, lse = s["layer"].step(s["q_idx"], s["w"], s["pool_key"], s["q"], s["kv"], s["kv_scale"], s["table"], s["npool"],
                               s["positions"], write=(s["rows"], s["ape"], s["slot_mapping"], s["rows_scale"]))
    return dict(out=out, lse=lse, pool_key=s["pool_key"])


def _run_chunk(s: dict) -> dict:
    i = s["inp"]
    c = i.cfg
    pools, cnt, vals = dsa_long_select.select(i.qI, i.w, i.k8, i.npool, c.keep, c.scale, pk_scale=i.k_scale,
                                              qI_scale=i.qI_scale)
    out, lse = dsa_decode.attend_tokens(i.q, i.kv_cache, i.kv_scale, pools, cnt, s["tables"], PAGE, c.softmax_scale)
    return dict(pools=pools, cnt=cnt, vals=vals, out=out, lse=lse)


def _run_pooled_chunk(s: dict) -> dict:
    i = s["inp"]
    c = i.cfg
    pools, cnt, vals = dsa_long_select.select(i.qI, i.w, i.pk, i.npool, c.keep, c.scale)
    out, lse = dsa_long.attend_pooled(i.q, i.kv_cache, i.kv_scale, pools, cnt, i.npool, i.positions, i.table, PAGE, KP,
                                      c.softmax_scale, lse=True)
    return dict(pools=pools, cnt=cnt, vals=vals, out=out, lse=lse)


def _run_store(s: dict) -> dict:
    dsa_cache.store(s["latent_cache"], s["slot_mapping"], s["latent"], scale=s["latent_scale"])
    dsa_cache.store(s["key_cache"], s["slot_mapping"], s["key"], scale=s["key_scale"])
    return dict(latent=s["latent_cache"].view(torch.uint8), latent_scale=s["latent_scale"],
                key=s["key_cache"].view(torch.uint8), key_scale=s["key_scale"])


def run(state: dict):
    return globals()["_run_" + state["case"]["family"]](state)


# -- what a pass cannot do without -------------------------------------------------------------------------------


def work(case: dict) -> dict:
    f = case["family"]
    if f == "decode":  # ragged batches: the mean length for all but the longest row
        B, L, H, Hi = case["B"], case["L"], case["H"], case["Hi"]
        n = [L] + [(case["low"] + L) // 2] * (B - 1)
        sel = sum(min(KEEP, x) for x in n)
        return dict(bytes=W.algorithmic_bytes(n, H, Hi, KEEP, PAGE) + 4 * B * H,
                    flops=2 * 128 * Hi * sum(n) + 2 * H * (576 + 512) * sel)
    if f == "pooled":
        B, L, H, Hi = case["B"], case["L"], case["H"], case["Hi"]
        n = [L] + [(case["low"] + L) // 2] * (B - 1)
        cfg = W.PooledConfig("case", B=B, L=L, H=H, Hi=Hi)
        tok = [min(KEEP, x) for x in n]
        return dict(bytes=W.pooled_step_bytes(cfg, [x // KP for x in n], tok) + 4 * B * H,
                    flops=2 * 128 * Hi * sum(x // KP for x in n) + 2 * H * (512 + 512) * sum(tok))
    if f == "store":
        T, e = case["T"], 4 if case["x_fp32"] else 2
        return dict(bytes=T * ((576 + 128) * (e + 1) + 2 * 4 + 8), flops=4 * T * (576 + 128))
    N, cached, H, Hi = case["N"], case["cached"], case["H"], case["Hi"]
    kp, dqk = (KP, 512) if f == "pooled_chunk" else (1, 576)
    cand = sum((cached + i + 1) // kp for i in range(N))
    tok = sum(min(KEEP, cached + i + 1) for i in range(N))
    P = (cached + N + kp - 1) // kp
    qb = 1 if case.get("q_fp8") else 2
    # every context row is attended by some query; the chunk's outputs, the selections and their scores
    nbytes = N * Hi * (128 * qb + 4) + P * (256 if kp > 1 else 132) + (cached + N) * (dqk + 4) + N * H * 2 * dqk
    nbytes += N * H * 512 * (4 if kp > 1 else 2) + N * (KEEP // kp) * 12 + N * 8
    return dict(bytes=nbytes, flops=2 * 128 * Hi * cand + 2 * H * (dqk + 512) * tok)


def tolerance(case: dict):
    if case["family"] == "store":
        return "exact"  # bytes and correctly rounded scales
    # out is bf16 and so are the softmax weights that it sums with (two orders of the sums differ by about 2.5e-3 of
    # it); a score within an fp32 rounding of the last selected one can change places with it, which shifts the
    # positions and scores listed after it in that row of a chunk's 64 to 2,048
    return dict(rel=1e-2, max=0.4, differ=0.01)


# -- the same in 64 bits -----------------------------------------------------------------------------------------


def _attend64(q, rows, scale):
    """q [H, D], rows [n, D] in 64 bits -> out [H, 512], lse [H]."""
    s = q @ rows.T.contiguous() * scale
    m = s.amax(1, keepdim=True)
    p = (s - m).exp()
    tot = p.sum(1, keepdim=True)
    return (p / tot) @ rows[:, :512].contiguous(), (m + tot.log()).squeeze(1)


def _scores64(q, w, k):
    """q [H, 128], w [H], k [n, 128] in 64 bits -> [n]."""
    return torch.cat([w @ torch.relu(q @ c.T.contiguous()) for c in k.split(131072)])


def _exact_decode(case: dict, seed: int) -> dict:
    s = prepare(case, seed)
    i = s["inp"]
    outs, lses = [], []
    for b, n in enumerate(i.lengths):
        t = torch.arange(n, device=DEV)
        slot = i.table[b].long()[t // PAGE] * PAGE + t % PAGE
        sc = torch.cat([_scores64(i.q_idx[b].double(), i.w_k[b].double(),
                                  i.k_cache[c].double() * i.k_scale[c].double().unsqueeze(1)) for c in slot.split(262144)])
        at = slot[sc.topk(min(KEEP, n)).indices]
        o, ls = _attend64(i.q[b].double(), i.kv_cache[at].double() * i.kv_scale[at].double().unsqueeze(1), s["layer"].scale)
        outs.append(o)
        lses.append(ls)
    return dict(out=torch.stack(outs), lse=torch.stack(lses))


def _pool_tokens(pools, npool: int, position: int):
    tok = (pools.view(-1, 1) * KP + torch.arange(KP, device=DEV)).view(-1)
    return torch.cat([tok, torch.arange(npool * KP, position + 1, device=DEV)])  # and the incomplete pool's


def _exact_pooled(case: dict, seed: int) -> dict:
    s = prepare(case, seed)
    outs, lses = [], []
    for b in range(case["B"]):
        pos, npool = int(s["positions"][b]), int(s["npool"][b])
        page = s["table"][b].long()
        if npool:
            p = torch.arange(npool, device=DEV)
            first = page[p * KP // PAGE] * PAGE + p * KP % PAGE
            keys = s["pool_key"][first.view(-1, 1) + torch.arange(KP, device=DEV)].reshape(npool, 128)
            sc = _scores64(s["q_idx"][b].double(), s["w"][b].double(), keys.double())
            pools = sc.topk(min(KEEP // KP, npool)).indices
        else:
            pools = torch.empty(0, dtype=torch.int64, device=DEV)
        t = _pool_tokens(pools, npool, pos)
        at = page[t // PAGE] * PAGE + t % PAGE
        o, ls = _attend64(s["q"][b].double(), s["kv"][at].double() * s["kv_scale"][at].double().unsqueeze(1), 256 ** -0.5)
        outs.append(o)
        lses.append(ls)
    return dict(out=torch.stack(outs), lse=torch.stack(lses), pool_key=None)  # pool_key: rounded to bf16 on the way


def _exact_rows(case: dict, seed: int, pooled: bool) -> dict:
    i = prepare(case, seed)["inp"]
    c = i.cfg
    kp = KP if pooled else 1
    keys = i.pk.double() if pooled else i.k8.double() * i.k_scale.double().unsqueeze(1)
    page = i.table.long()
    kT = keys.T.contiguous()
    outs, lses = [], []
    for n in range(case["N"]):
        m, pos = int(case["cached"] + n + 1) // kp, case["cached"] + n
        q = i.qI[n].double()
        if not pooled and i.qI_scale is not None:
            q = q * i.qI_scale[n].double().unsqueeze(1)
        sc = i.w[n].double() @ torch.relu(q @ kT[:, :m]) if m else torch.empty(0, dtype=torch.float64, device=DEV)
        top = sc.topk(min(KEEP // kp, m)).indices
        t = _pool_tokens(top, m, pos) if pooled else top
        at = page[t // PAGE] * PAGE + t % PAGE
        o, ls = _attend64(i.q[n].double(), i.kv_cache[at].double() * i.kv_scale[at].double().unsqueeze(1), c.softmax_scale)
        outs.append(o)
        lses.append(ls)
    # pools, cnt and vals: whole numbers, and scores listed by position, where one place changed shifts a row's rest
    return dict(pools=None, cnt=None, vals=None, out=torch.stack(outs), lse=torch.stack(lses))


def exact(case: dict, seed: int):
    f = case["family"]
    if f == "store":
        return None  # bytes: compared as they are
    if f in ("chunk", "pooled_chunk"):
        return _exact_rows(case, seed, f == "pooled_chunk")
    return _exact_decode(case, seed) if f == "decode" else _exact_pooled(case, seed)
