"""The work that users of the paged-KV library have it do, as cases to time.

An inference engine drives the library layer by layer: prompts come in as
chunks whose K/V rows are appended and attended causally (extend), every
engine step then decodes one token per running sequence from a plan built
once per step, pages are copied and moved when prefixes are shared or the
pool is compacted, and requests are handed between workers in the wire form.
Each case is one such piece of work at one size.

Shapes are those of the benchmark configurations (mitten_amd.workloads) and
one generic grouped-query geometry of 32 query and 8 KV heads. Layer counts
are cut where a full model would only repeat the same launches over more
memory. Lengths are a function of the case; contents and page tables of the
seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mitten_amd import DeviceKvPool, PoolDesc
from mitten_amd.device_pool import rope_inv_freq
from mitten_amd.workloads import CONFIGS

PAGE = 16
DEV = "cuda:0"
GEOMETRY = {name: (c["num_q_heads"], c["num_kv_heads"], c["head_dim"], c["dtype"]) for name, c in CONFIGS.items()}
GEOMETRY["gqa-32-8"] = (32, 8, 128, "bf16")
ROPE_THETA = 1e6


# ---- cases ------------------------------------------------------------------


def listed():
    return [
        # A small chat server on the f32 model: few short sequences, every
        # layer's grown KV state gathered for the caller. Launch latency.
        dict(name="decode_small_f32", kind="decode", model="qwen2.5-0.5b", layers=24, seqs=8, lo=33, hi=513, lens=1,
             gather=True),
        # One user with a long context: a few pages' worth of work per CU.
        dict(name="decode_one_long", kind="decode", model="qwen2.5-7b", layers=28, seqs=1, lo=8193, hi=8193, lens=2,
             gather=False),
        # The ordinary serving step: 64 ragged sequences.
        dict(name="decode_batch", kind="decode", model="qwen2.5-7b", layers=8, seqs=64, lo=1025, hi=8193, lens=3,
             gather=False),
        # Multi-query heads of dimension 256, a large batch.
        dict(name="decode_mqa", kind="decode", model="gemma-2b-mqa", layers=6, seqs=128, lo=2049, hi=8193, lens=4,
             gather=False),
        # A system prompt shared by every sequence through the radix cache.
        dict(name="decode_shared_prefix", kind="shared", model="qwen2.5-7b", layers=6, seqs=256, prefix=4096, lo=64,
             hi=1060, lens=5),
        # Decode without a plan: tables and lengths stay on the device.
        dict(name="attend_device_tables", kind="attend", model="gqa-32-8", layers=4, seqs=24, lo=300, hi=4100, lens=6),
        # Prefill chunks of long prompts: append and causal attention.
        dict(name="extend_chunks", kind="extend", model="qwen2.5-7b", layers=2, seqs=8, qlo=512, qhi=512, plo=4096,
             phi=4096, lens=7),
        # Short chunks over long contexts (multi-turn chat, draft checking).
        dict(name="extend_short", kind="extend", model="qwen2.5-7b", layers=4, seqs=16, qlo=5, qhi=24, plo=4000,
             phi=8000, lens=8),
        # Whole prompts of the f32 model.
        dict(name="extend_prompts_f32", kind="extend", model="qwen2.5-0.5b", layers=4, seqs=8, qlo=32, qhi=512, plo=0,
             phi=0, lens=9),
        # The step before attention: norm, rotary embedding and append.
        dict(name="prep_prefill", kind="prep", model="qwen2.5-7b", layers=2, tokens=16384, rotary=128, gated=True),
        # Compaction or copy-on-write: whole pages, every layer.
        dict(name="copy_pages", kind="copy", model="qwen2.5-7b", layers=28, pages=2069),
        # A request handed to another worker: export, then import.
        dict(name="wire_handoff", kind="wire", model="qwen2.5-7b", layers=28, pages=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "shared", "attend", "extend", "extend", "extend", "prep", "copy", "wire"])
    model = rng.choice(list(GEOMETRY))
    if kind in ("shared", "copy", "wire") and GEOMETRY[model][3] == "f32":
        model = "qwen2.5-7b"
    hq, hkv, d, dt = GEOMETRY[model]
    c = dict(kind=kind, model=model)
    if kind in ("decode", "attend"):
        c.update(layers=rng.choice([2, 4, 6]), seqs=_log(rng, 1, 128), lens=rng.randrange(1 << 20))
        c["hi"] = _log(rng, 33, 8193)
        c["lo"] = _log(rng, 1, c["hi"])
        if kind == "decode":
            c["gather"] = dt == "f32" and rng.random() < 0.5
        # K/V bytes of all layers stay below the listed batch's.
        row = 2 * hkv * d * (4 if dt == "f32" else 2) * c["layers"]
        c["seqs"] = max(1, min(c["seqs"], int(4e9 / (row * c["hi"]))))
    elif kind == "shared":
        c.update(layers=rng.choice([2, 4]), seqs=_log(rng, 8, 256), prefix=PAGE * _log(rng, 16, 400),
                 lens=rng.randrange(1 << 20))
        c["hi"] = _log(rng, 16, 1060)
        c["lo"] = _log(rng, 1, c["hi"])
    elif kind == "extend":
        f32 = dt == "f32"
        c.update(layers=rng.choice([1, 2, 4]), seqs=_log(rng, 1, 32), lens=rng.randrange(1 << 20))
        c["qhi"] = _log(rng, 2, 700 if f32 else 2048)
        c["qlo"] = _log(rng, 1, c["qhi"])
        c["phi"] = 0 if rng.random() < 0.4 else _log(rng, 1, 700 if f32 else 8000)
        c["plo"] = 0 if c["phi"] == 0 else _log(rng, 1, c["phi"])
        # Query-key pairs of all layers stay below a share of the listed chunks'.
        most = (2 if f32 else 40) * 1000 * 1000 * 28 * 128 / (hq * d)
        c["seqs"] = max(1, min(c["seqs"], int(most / (c["layers"] * c["qhi"] * (c["phi"] + c["qhi"])))))
    elif kind == "prep":
        c.update(layers=2, tokens=_log(rng, 1, 16384), gated=rng.random() < 0.5)
        c["rotary"] = d if rng.random() < 0.6 else d // 2
        c["tokens"] = max(1, min(c["tokens"], int(16384 * 28 * 128 * 2 / (hq * d * (4 if dt == "f32" else 2)))))
    else:
        row = 2 * hkv * d * 2 * PAGE
        c.update(layers=rng.choice([4, 18, 28]), pages=_log(rng, 1, 2069 if kind == "copy" else 512))
        c["pages"] = max(1, min(c["pages"], int((1.8e9 if kind == "copy" else 2.2e8) / (row * c["layers"]))))
    return c


# ---- inputs (the same from prepare and exact) ---------------------------------


def _dtype(case):
    return torch.float32 if GEOMETRY[case["model"]][3] == "f32" else torch.bfloat16


def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + part) % (1 << 62))


def _normal(shape, case, seed, part, scale=1.0):
    t = torch.empty(shape, dtype=_dtype(case), device=DEV)
    t.normal_(0.0, scale, generator=_gen(seed, part))
    return t


def _lens(case, lo, hi, part=0):
    return np.random.default_rng([case["lens"], part]).integers(case[lo], case[hi] + 1, size=case["seqs"])


def _tables(nblk, seed, front=0):
    """CSR page tables of nblk[b] pages each, slices of a permutation of the
    pool; the first `front` ids of the permutation go to nobody."""
    nblk = np.asarray(nblk, np.int64)
    total = int(nblk.sum()) + front
    perm = np.random.default_rng(int(seed)).permutation(total).astype(np.uint32)
    indptr = np.zeros(nblk.size + 1, np.uint32)
    indptr[1:] = np.cumsum(nblk)
    return total, indptr, perm[front:].copy(), perm[:front].copy()


def _pages(tokens):
    return (np.asarray(tokens, np.int64) + PAGE - 1) // PAGE


class _PoolView:
    """What keeps the pool alive for as long as a tensor over its buffer is."""

    def __init__(self, pool, typestr):
        self.pool = pool
        self.__cuda_array_interface__ = {"shape": tuple(int(x) for x in pool.desc.shape), "typestr": typestr,
                                         "data": (pool.data_ptr, False), "version": 3, "strides": None}


def _pool(case, blocks):
    hq, hkv, d, dt = GEOMETRY[case["model"]]
    pool = DeviceKvPool(PoolDesc(case["layers"], hkv, hq, d, int(blocks), dtype=dt))
    t = torch.as_tensor(_PoolView(pool, "<f4" if dt == "f32" else "<i2"), device=DEV)
    return pool, t if dt == "f32" else t.view(torch.bfloat16)


def _content(case, blocks, seed, out=None):
    """K/V that earlier steps left in the pool: [layers][2][blocks][16][heads][dim]."""
    hq, hkv, d, _ = GEOMETRY[case["model"]]
    if out is None:
        out = torch.empty((case["layers"], 2, int(blocks), PAGE, hkv, d), dtype=_dtype(case), device=DEV)
    return out.normal_(generator=_gen(seed, 1))


def _bits(t):
    """K/V that were moved, not computed: compared as whole numbers."""
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)


def _slots(ids, indptr, b, pos):
    return ids[indptr[b] + pos // PAGE].astype(np.uint32) * PAGE + (pos % PAGE).astype(np.uint32)


Q_SCALE = 1.5  # queries: scores of standard deviation 1.5, some keys well above the rest


def _decode_inputs(case, seed, lens):
    hq, hkv, d, _ = GEOMETRY[case["model"]]
    L, B = case["layers"], len(lens)
    return (_normal((L, B, hkv, d), case, seed, 2), _normal((L, B, hkv, d), case, seed, 3),
            _normal((L, B, hq, d), case, seed, 4, Q_SCALE))


def _extend_inputs(case, seed):
    hq, hkv, d, _ = GEOMETRY[case["model"]]
    ql = _lens(case, "qlo", "qhi")
    ctx = _lens(case, "plo", "phi", 1) + ql
    blocks, ip, ids, _ = _tables(_pages(ctx), seed)
    slots = np.concatenate([_slots(ids, ip, b, np.arange(ctx[b] - ql[b], ctx[b])) for b in range(len(ql))])
    L, T = case["layers"], int(ql.sum())
    return (ql, ctx, blocks, ip, ids, slots, _normal((L, T, hkv, d), case, seed, 2),
            _normal((L, T, hkv, d), case, seed, 3), _normal((L, T, hq, d), case, seed, 4, Q_SCALE))


def _prep_inputs(case, seed):
    hq, hkv, d, _ = GEOMETRY[case["model"]]
    L, n = case["layers"], case["tokens"]
    blocks, _, ids, _ = _tables([int(_pages(n))], seed)
    pos = np.arange(n)
    slots = ids[pos // PAGE].astype(np.uint32) * PAGE + (pos % PAGE).astype(np.uint32)
    w = [torch.randn(d, generator=_gen(seed, 6 + i), device=DEV) * 0.1 for i in range(2)]
    inv = torch.from_numpy(rope_inv_freq(case["rotary"], ROPE_THETA)).to(DEV)
    qshape = (L, n, hq, 2, d) if case["gated"] else (L, n, hq, d)
    return (blocks, slots, (pos + 100).astype(np.int32), w, inv, _normal(qshape, case, seed, 2, 2.0),
            _normal((L, n, hkv, d), case, seed, 3, 2.0), _normal((L, n, hkv, d), case, seed, 4))


# ---- prepare and run ------------------------------------------------------------


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_decode(case, seed):
    hq, hkv, d, _ = GEOMETRY[case["model"]]
    ctx = _lens(case, "lo", "hi").astype(np.int32)
    blocks, ip, ids, _ = _tables(_pages(ctx), seed)
    pool, view = _pool(case, blocks)
    _content(case, blocks, seed, view)
    k, v, q = _decode_inputs(case, seed, ctx)
    out = torch.empty_like(q)
    plan = pool.plan(ctx, block_indptr=ip, block_ids=ids)
    g = None
    if case["gather"]:
        n = int(ctx.sum()) * hkv * d
        g = tuple(torch.zeros(n, dtype=_dtype(case), device=DEV) for _ in range(2))
    step = pool.bind_decode_step(plan, k, v, q, None, None, out, gather_out=g)
    outputs = {"o": out, "pool": _bits(view)}
    if g is not None:
        outputs.update(gather_k=_bits(g[0]), gather_v=_bits(g[1]))
    return dict(run=_run_decode, pool=pool, plan=plan, ctx=ctx, ip=ip, ids=ids, step=step, layers=case["layers"],
                outputs=outputs)


def _run_decode(s):
    # One engine step: the plan from the scheduler's lengths and tables, then every layer.
    s["plan"].build(s["ctx"], 0, None, s["ip"], s["ids"])
    for layer in range(s["layers"]):
        s["step"](layer)
    return s["outputs"]


def _prepare_shared(case, seed):
    suf = _lens(case, "lo", "hi").astype(np.int32)
    blocks, ip, ids, pre = _tables(_pages(suf), seed, case["prefix"] // PAGE)
    pool, view = _pool(case, blocks)
    _content(case, blocks, seed, view)
    k, v, q = _decode_inputs(case, seed, suf)
    out = torch.empty_like(q)
    plan = pool.plan_shared_prefix(pre, suf, ip, ids)
    step = pool.bind_decode_step_shared_prefix(plan, k, v, q, None, None, None, out)
    return dict(run=_run_shared, pool=pool, plan=plan, suf=suf, ip=ip, ids=ids, pre=pre, step=step,
                layers=case["layers"], outputs={"o": out, "pool": _bits(view)})


def _run_shared(s):
    s["plan"].build(s["suf"], 0, None, s["ip"], s["ids"], s["pre"])
    for layer in range(s["layers"]):
        s["step"](layer)
    return s["outputs"]


def _prepare_attend(case, seed):
    ctx = _lens(case, "lo", "hi").astype(np.int32)
    blocks, ip, ids, _ = _tables(_pages(ctx), seed)
    pool, view = _pool(case, blocks)
    _content(case, blocks, seed, view)
    _, _, q = _decode_inputs(case, seed, ctx)
    dev = [torch.from_numpy(np.asarray(a, np.int32)).to(DEV) for a in (ip, ids, ctx)]
    return dict(run=_run_attend, pool=pool, view=view, q=list(q), out=list(torch.empty_like(q)), dev=dev,
                max_ctx=int(ctx.max()))


def _run_attend(s):
    ip, ids, ctx = s["dev"]
    return [s["pool"].decode_attention(layer, q, ip, ids, ctx, s["max_ctx"], out=s["out"][layer])
            for layer, q in enumerate(s["q"])]


def _prepare_extend(case, seed):
    ql, ctx, blocks, ip, ids, slots, k, v, q = _extend_inputs(case, seed)
    pool, view = _pool(case, blocks)
    _content(case, blocks, seed, view)
    out = torch.empty_like(q)
    return dict(run=_run_extend, pool=pool, ql=ql.astype(np.int32), ctx=ctx.astype(np.int32), ip=ip, ids=ids,
                slots=slots, layers=list(zip(k, v, q, out)), outputs={"o": out, "pool": _bits(view)})


def _run_extend(s):
    pool = s["pool"]
    for layer, (k, v, q, out) in enumerate(s["layers"]):
        pool.append(layer, k, v, s["slots"])
        pool.extend_attention_host(layer, q, s["ql"], s["ctx"], s["ip"], s["ids"], out=out)
    return s["outputs"]


def _prepare_prep(case, seed):
    blocks, slots, pos, w, inv, q, k, v = _prep_inputs(case, seed)
    pool, view = _pool(case, blocks)
    view.zero_()
    hq, _, d, _ = GEOMETRY[case["model"]]
    out = torch.empty((case["layers"], case["tokens"], hq, d), dtype=_dtype(case), device=DEV)
    return dict(run=_run_prep, pool=pool, slots=slots, pos=pos, w=w, inv=inv, gated=case["gated"],
                layers=list(zip(q, k, v, out)), outputs={"q": out, "pool": view})


def _run_prep(s):
    for layer, (q, k, v, out) in enumerate(s["layers"]):
        s["pool"].qk_norm_rope_append(layer, q, k, v, s["pos"], s["slots"], s["w"][0], s["w"][1], s["inv"],
                                      gated=s["gated"], out=out)
    return s["outputs"]


def _prepare_copy(case, seed):
    n = case["pages"]
    pool, view = _pool(case, 2 * n)
    _content(case, 2 * n, seed, view)
    perm = np.random.default_rng(int(seed)).permutation(2 * n).astype(np.uint32)
    return dict(run=_run_copy, pool=pool, src=perm[:n].copy(), dst=perm[n:].copy(), out=_bits(view))


def _run_copy(s):
    s["pool"].copy_blocks(s["src"], s["dst"])
    return s["out"]


def _prepare_wire(case, seed):
    n = case["pages"]
    pool, view = _pool(case, 2 * n)
    _content(case, 2 * n, seed, view)
    perm = np.random.default_rng(int(seed)).permutation(2 * n).astype(np.uint32)
    payload = torch.empty(n * pool.wire_block_bytes(), dtype=torch.uint8, device=DEV)
    sums = [torch.zeros(n, dtype=torch.int64, device=DEV) for _ in range(2)]
    return dict(run=_run_wire, pool=pool, src=perm[:n].copy(), dst=perm[n:].copy(), payload=payload, sums=sums,
                outputs={"payload": payload, "sent": sums[0], "received": sums[1], "pool": _bits(view)})


def _run_wire(s):
    s["pool"].wire_export(s["src"], payload=s["payload"], checksums=s["sums"][0])
    s["pool"].wire_import(s["dst"], s["payload"], expected=s["sums"][0], checksums=s["sums"][1])
    return s["outputs"]


# ---- what a pass cannot do without -----------------------------------------------


def work(case):
    hq, hkv, d, dt = GEOMETRY[case["model"]]
    es, L, kind = (4 if dt == "f32" else 2), case["layers"], case["kind"]
    kv, qo = 2 * hkv * d * es, 2 * hq * d * es  # a token's K and V rows; a query row and its output
    if kind in ("decode", "attend"):
        ctx = _lens(case, "lo", "hi")
        T, B = int(ctx.sum()), len(ctx)
        nbytes = T * kv + B * qo + 4 * int(_pages(ctx).sum()) + 8 * B
        if kind == "decode":
            nbytes += B * kv  # the step's new rows written
            if case["gather"]:
                nbytes += T * kv
        return {"bytes": L * nbytes, "flops": L * 4 * hq * d * T}
    if kind == "shared":
        suf = _lens(case, "lo", "hi")
        T, B = int(suf.sum()) + case["prefix"], len(suf)
        pairs = int(suf.sum()) + B * case["prefix"]
        return {"bytes": L * (T * kv + B * (qo + kv)), "flops": L * 4 * hq * d * pairs}
    if kind == "extend":
        ql = _lens(case, "qlo", "qhi")
        ctx = _lens(case, "plo", "phi", 1) + ql
        T = int(ql.sum())
        pairs = int((ql * ctx - ql * (ql - 1) // 2).sum())
        return {"bytes": L * (int(ctx.sum()) * kv + T * kv + T * qo), "flops": L * 4 * hq * d * pairs}
    if kind == "prep":
        n = case["tokens"]
        return {"bytes": L * n * (2 * kv + qo + 8), "flops": L * n * (hq + hkv) * d * 8}
    n = case["pages"]
    moved = 2 * n * PAGE * kv * L  # read once and written once
    return {"bytes": moved if kind == "copy" else 2 * moved, "flops": 0}


def tolerance(case):
    """Moved bytes and checksums are whole numbers and have to be the same.
    Attention and the norm are sums in 32 bits, rounded to the pool's type."""
    if case["kind"] in ("copy", "wire"):
        return "exact"
    if GEOMETRY[case["model"]][3] == "f32":
        # Rotary angles of position times frequency are rounded to 32 bits.
        return {"rel": 2e-4, "max": 1e-2} if case["kind"] == "prep" else {"rel": 4e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.1}


# ---- the same in 64 bits -----------------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    if kind in ("copy", "wire"):
        return None  # moved bytes: whole numbers
    with torch.no_grad():
        return globals()["_exact_" + kind](case, seed)


def _attend64(k, v, q, first):
    """q [n][Hq][D] at positions first .. first + n - 1 over k, v [ctx][Hkv][D]:
    query i sees keys 0 .. first + i."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    k, v = (t.double().transpose(0, 1).contiguous() for t in (k, v))
    scale = float(np.float32(d ** -0.5))
    q = q.double().reshape(n, hkv, hq // hkv, d)
    keys = torch.arange(k.shape[1], device=q.device)
    out = torch.empty_like(q)
    rows = max(1, int(2e8 // (k.shape[1] * (hq // hkv))))
    for h in range(hkv):
        kt = k[h].t().contiguous()
        for i in range(0, n, rows):
            s = torch.matmul(q[i:i + rows, h].reshape(-1, d), kt).reshape(-1, hq // hkv, k.shape[1]) * scale
            last = first + torch.arange(i, i + s.shape[0], device=q.device)
            s.masked_fill_(keys[None, None, :] > last[:, None, None], -math.inf)
            p = torch.softmax(s, -1)
            out[i:i + rows, h] = torch.matmul(p.reshape(-1, k.shape[1]), v[h]).reshape(-1, hq // hkv, d)
    return out.reshape(n, hq, d)


def _rows(content, layer, kv, ids, n):
    hkv, d = content.shape[-2:]
    at = torch.from_numpy(ids.astype(np.int64)).to(content.device)
    return content[layer, kv].index_select(0, at).reshape(-1, hkv, d)[:n].clone()


def _exact_decode(case, seed):
    ctx = _lens(case, "lo", "hi")
    blocks, ip, ids, pre = _tables(_pages(ctx), seed, case.get("prefix", 0) // PAGE)
    content = _content(case, blocks, seed)
    k_new, v_new, q = _decode_inputs(case, seed, ctx)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    gathered = [[], []]
    for layer in range(case["layers"]):
        for b, n in enumerate(int(x) for x in ctx):
            full = np.concatenate([pre, ids[ip[b]:ip[b + 1]]])
            n += case.get("prefix", 0)
            k, v = (_rows(content, layer, kv, full, n) for kv in (0, 1))
            if case["kind"] != "attend":
                k[n - 1], v[n - 1] = k_new[layer, b], v_new[layer, b]
            out[layer, b] = _attend64(k, v, q[layer, b:b + 1], n - 1)[0]
            if case.get("gather") and layer == case["layers"] - 1:
                for kv, t in enumerate((k, v)):
                    gathered[kv].append(t.transpose(0, 1).reshape(-1))
    if case["kind"] == "attend":
        return list(out)
    r = {"o": out, "pool": None}
    if case.get("gather"):
        r.update(gather_k=_bits(torch.cat(gathered[0])), gather_v=_bits(torch.cat(gathered[1])))
    return r


_exact_shared = _exact_attend = _exact_decode


def _exact_extend(case, seed):
    ql, ctx, blocks, ip, ids, _, k_new, v_new, q = _extend_inputs(case, seed)
    content = _content(case, blocks, seed)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    start = np.concatenate([[0], np.cumsum(ql)])
    for layer in range(case["layers"]):
        for b in range(len(ql)):
            n, first, rows = int(ctx[b]), int(ctx[b] - ql[b]), slice(int(start[b]), int(start[b + 1]))
            k, v = (_rows(content, layer, kv, ids[ip[b]:ip[b + 1]], n) for kv in (0, 1))
            k[first:], v[first:] = k_new[layer, rows], v_new[layer, rows]
            out[layer, rows] = _attend64(k, v, q[layer, rows], first)
    return {"o": out, "pool": None}


def _exact_prep(case, seed):
    blocks, slots, pos, w, inv, q, k, v = _prep_inputs(case, seed)
    hkv, d = k.shape[-2:]
    half = case["rotary"] // 2
    a = torch.from_numpy(pos).to(DEV).double()[:, None] * inv.double()[None, :]
    cos, sin = a.cos()[:, None, :], a.sin()[:, None, :]

    def normed(x, weight):
        x = x.double()
        x = x * (x.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (1.0 + weight.double())
        lo, hi, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin, rest], -1)

    if case["gated"]:
        q = q[:, :, :, 0]
    pool = torch.zeros((case["layers"], 2, blocks * PAGE, hkv, d), dtype=torch.float64, device=DEV)
    at = torch.from_numpy(slots.astype(np.int64)).to(DEV)
    out = []
    for layer in range(case["layers"]):
        out.append(normed(q[layer], w[0]))
        pool[layer, 0].index_copy_(0, at, normed(k[layer], w[1]))
        pool[layer, 1].index_copy_(0, at, v[layer].double())
    return {"q": torch.stack(out), "pool": pool.reshape(case["layers"], 2, blocks, PAGE, hkv, d)}
