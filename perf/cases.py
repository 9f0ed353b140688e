"""The work a program gives this package, as timed cases.

A case is one pass through the public entry points at one shape:

* ``step``    ``compute_hybrid_attention`` over one ``CompressedKVStore`` (a
              decode step with one query token, or a chunk of causal queries);
* ``batch``   a decode step over ``QuantizedKVBatch`` through its plan;
* ``paged``   a decode step over ``PagedQuantizedKV`` through its plan;
* ``encode``  the key codec and the value packer over [seqs, tokens, heads];
* ``append``  a chunk appended to an empty ``CompressedKVStore``;
* ``cache``   scores, softmax and ``attend`` of the standalone ``SMAQKVCache``.

Keys follow N(0, U diag(1/i) U^T) in a seeded random basis U; values and
queries N(0, 1).  Paged keys are heavy-tailed (Student-t, 3 degrees of
freedom), 2-dim block-VQ keys have four outlier channels times 20.
"""

from __future__ import annotations

import functools
import math

import torch

D = 128
VALUE_GROUP = 32
RING = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
OUTLIERS = (17, 40, 77, 101)

_BASE = dict(codec="scalar", key_bits=3, block_dim=0, value_bits=2, dtype="bf16", q_heads=32, kv_heads=8, seqs=1,
             tokens=0, recent=0, queries=1)


def _case(name, kind, **kw):
    c = dict(_BASE, kind=kind, **kw)
    if c["codec"] == "vq":
        c["key_bits"] = 0
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user's chat early on: a step is all launches and host work
        _case("step_short", "step", tokens=500, recent=37),
        # decode over a full batch of long contexts (32 x 32768, 32/8 heads)
        _case("batch_long", "batch", seqs=32, tokens=32768),
        # decode over the cache that encode_vq8 makes: 1 bit per key dim
        _case("batch_vq8", "batch", codec="vq", block_dim=8, seqs=16, tokens=32768),
        # paged serving: 256 sequences of up to 16384 tokens, 16-token blocks
        _case("paged_ragged", "paged", seqs=256, tokens=16384),
        # the same serving loop at 28/4 heads with fewer, shorter sequences
        _case("paged_gqa7", "paged", seqs=64, tokens=8000, q_heads=28, kv_heads=4),
        # the decode steps that follow chunk_long: one sequence, 65536 tokens
        _case("step_vq2_long", "step", codec="vq", block_dim=2, dtype="fp16", q_heads=28, kv_heads=4, tokens=65408,
              recent=128),
        # chunked prefill of a long prompt: 2048 causal queries
        _case("chunk_long", "step", codec="vq", block_dim=2, dtype="fp16", q_heads=28, kv_heads=4, tokens=65408,
              recent=128, queries=2048),
        # a few drafted tokens checked at once, in the first layers' 4-bit keys
        # and with 4-bit values
        _case("chunk_draft", "step", key_bits=4, value_bits=4, tokens=4001, recent=100, queries=5),
        # a whole cache encoded at 1 bit per key dim, 2-bit values
        _case("encode_vq8", "encode", codec="vq", block_dim=8, seqs=16, tokens=32768),
        # the long prompt's history encoded at 4 bits per key dim
        _case("append_vq2", "append", codec="vq", block_dim=2, dtype="fp16", q_heads=28, kv_heads=4, tokens=65408),
        # an ordinary prompt encoded, an odd number of tokens
        _case("append_scalar", "append", tokens=2047),
        # the standalone cache's decode step in fp32
        _case("cache_step", "cache", dtype="fp32", q_heads=8, kv_heads=8, seqs=2, tokens=8192),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(("step", "step", "batch", "batch", "paged", "chunk", "chunk", "encode", "append", "cache"))
    kw = {}
    if kind == "cache" or rng.random() < 0.6:
        kw.update(codec="scalar", key_bits=rng.choice((3, 3, 4)))
    else:
        kw.update(codec="vq", block_dim=rng.choice((2, 8)))
    kw["q_heads"], kw["kv_heads"] = rng.choice(((32, 8), (28, 4), (8, 8)))
    kw["dtype"] = rng.choice(("bf16", "bf16", "fp16"))
    kw["value_bits"] = rng.choice((2, 2, 4))
    hkv = kw["kv_heads"]
    if kind == "step":
        if kw["codec"] == "scalar" and rng.random() < 0.25:
            kw["dtype"] = "fp32"
        return _case("", "step", tokens=_log(rng, 16, 65408), recent=rng.randint(0, RING), **kw)
    if kind == "chunk":
        tokens = _log(rng, 500, 65408)
        return _case("", "step", tokens=tokens, recent=rng.randint(0, RING), queries=_log(rng, 2, min(2048, tokens)),
                     **kw)
    if kind == "batch":
        seqs = _log(rng, 2, 64)
        most = (8 if kw["codec"] == "scalar" else 4) * (1 << 20) // (seqs * hkv)
        return _case("", "batch", seqs=seqs, tokens=_log(rng, 300, min(32768, most)), **kw)
    if kind == "paged":
        seqs = _log(rng, 4, 256)
        return _case("", "paged", seqs=seqs, tokens=_log(rng, 600, min(16384, (1 << 22) // (seqs * hkv) * 2)), **kw)
    if kind == "cache":
        kw.update(q_heads=hkv, dtype="fp32")
        return _case("", "cache", seqs=rng.randint(1, 4), tokens=_log(rng, 300, 16384), **kw)
    if kind == "append":
        return _case("", "append", tokens=_log(rng, 16, 65408), **kw)
    return _case("", "encode", seqs=rng.randint(1, 16), tokens=_log(rng, 300, 16384), **kw)


# ------------------------------------------------------------ calibration ---

def _shaping(sigma, c=5.0):
    """E, E_inv of a covariance: its log-compressed, volume-normalised spectrum."""
    lam, vec = torch.linalg.eigh(sigma)
    logs = torch.log(torch.log1p(c * lam.clamp(min=0)).clamp(min=1e-8))
    s = torch.exp(logs - logs.mean())
    return vec @ torch.diag(s.sqrt()) @ vec.T, vec @ torch.diag(1.0 / s.sqrt()) @ vec.T


@functools.lru_cache(maxsize=None)
def _basis():
    """(Sigma, mix): Sigma = U diag(1/i) U^T and z @ mix ~ N(0, Sigma), on the CPU."""
    a = torch.randn(D, D, generator=torch.Generator().manual_seed(0), dtype=torch.float64)
    u, r = torch.linalg.qr(a)
    u = u * torch.sign(torch.diagonal(r))
    lam = 1.0 / torch.arange(1, D + 1, dtype=torch.float64)
    return ((u * lam) @ u.T).float(), (u * lam.sqrt()).T.float().contiguous()


@functools.lru_cache(maxsize=None)
def _codebook(block_dim):
    """A model's block-VQ calibration: (E, E_inv, centroids, decoded) per block,
    from sampled keys and a few Lloyd iterations, on the CPU."""
    g = torch.Generator().manual_seed(5)
    keys, queries = (torch.randn(4096, D, generator=g) @ _basis()[1] for _ in range(2))
    if block_dim == 2:
        keys[:, OUTLIERS] *= 20
    tables = []
    for b in range(D // block_dim):
        sl = slice(b * block_dim, (b + 1) * block_dim)
        E, E_inv = _shaping(queries[:, sl].T @ queries[:, sl] / queries.shape[0])
        x = keys[:, sl] @ E.T
        cents = x[torch.randperm(x.shape[0], generator=g)[:256]].clone()
        for _ in range(3):
            hit = torch.nn.functional.one_hot(torch.cdist(x, cents).argmin(1), 256).float()
            n = hit.sum(0).unsqueeze(1)
            cents = torch.where(n > 0, hit.T @ x / n.clamp(min=1), cents)
        tables.append((E, E_inv, cents, cents @ E_inv.T))
    return tuple(torch.stack(t) for t in zip(*tables))


@functools.lru_cache(maxsize=None)
def _scalar_tables(bits):
    """(centroids, inner boundaries): Gaussian quantiles in fp32."""
    def ppf(p):
        return math.sqrt(2.0) * torch.erfinv(2.0 * p - 1.0)
    cents = ppf(torch.linspace(0.0, 1.0, 2 ** bits + 2)[1:-1])
    return cents, ppf(torch.linspace(0.0, 1.0, 2 ** bits + 1).clamp(1e-6, 1.0 - 1e-6))[1:-1]


def _strategy(case):
    import smaq_amd as S
    if case["codec"] == "scalar":
        return S.SMAQFullMetricScalarStrategy(D, bits=case["key_bits"], Sigma_q=_basis()[0], device="cuda")
    strat = S.SMAQBlockVQStrategy(D, block_dim=case["block_dim"], n_centroids=256, device="cuda")
    E, E_inv, cents, decoded = _codebook(case["block_dim"])
    strat.quantizer.load_state_dict({"E_blocks": E, "E_inv_blocks": E_inv, "centroids": cents,
                                     "decoded_centroids": decoded})
    return strat


# ----------------------------------------------------------------- inputs ---

def _generator(seed, stream):
    return torch.Generator(device="cuda").manual_seed(1009 * int(seed) + stream)


def _keys(case, shape, seed, stream):
    """[*shape, D] keys in the case's dtype."""
    g, dt = _generator(seed, stream), DTYPES[case["dtype"]]
    n = math.prod(shape)
    mix = _basis()[1].cuda()
    out = torch.empty(n, D, dtype=dt, device="cuda")
    for i in range(0, n, 1 << 21):
        m = min(n, i + (1 << 21)) - i
        if case["kind"] == "paged":
            k = torch.randn(m, D, generator=g, device="cuda")
            chi = torch.zeros_like(k)
            for _ in range(3):
                chi += torch.randn(m, D, generator=g, device="cuda").square()
            k = k / (chi / 3).sqrt()
        else:
            k = torch.randn(m, D, generator=g, device="cuda") @ mix
            if case["block_dim"] == 2:
                k[:, OUTLIERS] *= 20
        out[i:i + m] = k.to(dt)
    if case["dtype"] == "fp32" and stream == 1:
        # no key whose code the order of a 32-bit sum could decide
        y = _scalar_units(out) @ _shaping(_basis()[0])[0].cuda().double().T
        b = _scalar_tables(case["key_bits"])[1].cuda().double()
        near = torch.stack([(y - x).abs().amin(1) for x in b]).amin(0) < 4e-6
        good = (~near).nonzero().flatten()
        out[near] = out[good[:int(near.sum())]]
    return out.view(*shape, D)


def _randn(case, shape, seed, stream):
    return torch.randn(*shape, D, generator=_generator(seed, stream), device="cuda").to(DTYPES[case["dtype"]])


def _queries(case, shape, seed):
    """Queries: of the keys' own covariance for block-VQ caches, else N(0, 1)."""
    if case["codec"] == "vq":
        z = torch.randn(*shape, D, generator=_generator(seed, 3), device="cuda")
        return (z @ _basis()[1].cuda()).to(DTYPES[case["dtype"]])
    return _randn(case, shape, seed, 3)


def _lengths(case, seed):
    """Ragged lengths, tokens / 16 to tokens."""
    g = torch.Generator().manual_seed(1009 * int(seed) + 7)
    return torch.randint(case["tokens"] // 16, case["tokens"] + 1, (case["seqs"],), generator=g).tolist()


def _tokens_in(case, seed):
    """(keys, values) of the whole case: [rows..., kv_heads, D]."""
    h = case["kv_heads"]
    if case["kind"] == "paged":
        shape = (sum(_lengths(case, seed)), h)
    elif case["kind"] == "cache":
        shape = (case["seqs"], h, case["tokens"])
    elif case["kind"] in ("batch", "encode"):
        shape = (case["seqs"], case["tokens"], h)
    else:
        shape = (case["tokens"], h)
    return _keys(case, shape, seed, 1), _randn(case, shape, seed, 2)


def _recent(case, seed):
    if not case["recent"]:
        return None, None
    shape = (case["recent"], case["kv_heads"])
    return _keys(case, shape, seed, 4), _randn(case, shape, seed, 5)


def _positions(case):
    """Causal positions of a chunk: its queries are the context's last tokens."""
    total = case["tokens"] + case["recent"]
    if case["queries"] == 1:
        return None
    return torch.arange(total - case["queries"], total, device="cuda")


def prepare(case, seed):
    import smaq_amd as S
    from smaq_amd.batch import PagedQuantizedKV, QuantizedKVBatch
    kind, hq, h, bits = case["kind"], case["q_heads"], case["kv_heads"], case["value_bits"]
    strat = _strategy(case)
    keys, values = _tokens_in(case, seed)
    state = dict(case=case, strat=strat)
    if kind == "encode":
        return dict(state, keys=keys, values=values)
    if kind == "append":
        store = S.CompressedKVStore(D, h, value_bits=bits, value_group_size=VALUE_GROUP, device="cuda",
                                    key_strategy=strat)
        return dict(state, store=store, keys=keys, values=values)
    if kind == "cache":
        cache = S.SMAQKVCache(D, value_bits=bits, value_group_size=VALUE_GROUP, buffer_size=RING, device="cuda",
                              dtype=torch.float32, key_strategy=strat)
        cache.prefill(keys, values)
        return dict(state, cache=cache, q=_queries(case, (case["seqs"], h, 1), seed))
    if kind == "step":
        store = S.CompressedKVStore(D, h, value_bits=bits, value_group_size=VALUE_GROUP, device="cuda",
                                    key_strategy=strat)
        store.append_chunk(keys, values)
        rk, rv = _recent(case, seed)
        return dict(state, store=store, rk=rk, rv=rv, q=_queries(case, (case["queries"], hq), seed),
                    pos=_positions(case))
    q = _queries(case, (case["seqs"], hq), seed)
    if kind == "batch":
        kv = QuantizedKVBatch.encode(strat, keys, values, value_bits=bits, value_group=VALUE_GROUP)
    else:
        lens = _lengths(case, seed)
        nblk = [-(-n // 16) for n in lens]
        g = torch.Generator().manual_seed(1009 * int(seed) + 8)
        perm = torch.randperm(sum(nblk), generator=g).to(torch.int32)
        table = torch.zeros(len(lens), max(nblk), dtype=torch.int32)
        at = 0
        for b, n in enumerate(nblk):
            table[b, :n] = perm[at:at + n]
            at += n
        kv = PagedQuantizedKV.encode(strat, keys.split(lens), values.split(lens), table.cuda(), sum(nblk),
                                     block_size=16, value_bits=bits, value_group=VALUE_GROUP)
    return dict(state, q=q, kv=kv, plan=kv.plan(q))


def run(state):
    from smaq_amd import compute_hybrid_attention, quantize_values
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        return compute_hybrid_attention(state["q"], state["store"], state["rk"], state["rv"], case["q_heads"],
                                        query_positions=state["pos"])
    if kind in ("batch", "paged"):
        return state["plan"].run(state["q"])
    if kind == "cache":
        scores = state["cache"].attention_scores(state["q"])
        return scores, state["cache"].attend(torch.softmax(scores, dim=-1))
    if kind == "encode":
        kq = state["strat"].quantize(state["keys"])
        vq = quantize_values(state["values"], bits=case["value_bits"], group_size=VALUE_GROUP)
    else:
        state["store"].reset()
        state["store"].append_chunk(state["keys"], state["values"])
        flat = state["store"].get_flat_cache()
        kq, vq = flat.key_q, flat.value_q
    return {"codes": kq.indices, "norms": getattr(kq, "norms", None), "data": vq.data, "scales": vq.scales,
            "zeros": vq.zeros}


# ------------------------------------------------------------------- work ---

def _key_bytes(case):
    if case["codec"] == "vq":
        return D // case["block_dim"]
    return D // 2 + torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()


def _row_bytes(case):
    """Bytes of one token-head: key codes, norm, value codes, scales, zeros."""
    es = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    return _key_bytes(case) + D * case["value_bits"] // 8 + 2 * (D // VALUE_GROUP) * es


def work(case):
    es = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    h, hq, n, b, t = case["kv_heads"], case["q_heads"], case["tokens"], case["seqs"], case["queries"]
    if case["kind"] in ("encode", "append"):
        rows = b * n * h
        flops = 2 * D * (D if case["codec"] == "scalar" else case["block_dim"] + 256)
        return {"bytes": rows * (2 * D * es + _row_bytes(case)), "flops": rows * flops}
    if case["kind"] == "cache":
        hist, recent = b * h * (n - RING), b * h * RING
    elif case["kind"] == "paged":
        hist, recent = sum(_lengths(case, 1)) * h, 0
    else:
        hist, recent = b * h * n, b * h * case["recent"]
    pairs = (hist + recent) * (hq // h) * t
    if t > 1:
        pairs -= hq * (t * (t - 1) // 2)
    return {"bytes": hist * _row_bytes(case) + recent * 2 * D * es + 2 * b * t * hq * D * es, "flops": 4 * D * pairs}


def tolerance(case):
    if case["kind"] in ("encode", "append"):
        return "exact"
    return {"bf16": {"rel": 8e-3}, "fp16": {"rel": 1.5e-3}, "fp32": {"rel": 1e-5}}[case["dtype"]]


# ---------------------------------------------------------------- exact -----

def _scalar_units(rows):
    """Rows over their norms, both in the rows' dtype, as float64."""
    n = rows.double().norm(dim=-1).to(rows.dtype)
    return (rows.float() / n.float().unsqueeze(-1)).to(rows.dtype).double()


def _decoded_keys(case, keys):
    """What the codec keeps of keys [..., D], in 64 bits."""
    rows = keys.reshape(-1, D)
    out = torch.empty(rows.shape, dtype=torch.float64, device=rows.device)
    step = 1 << (20 if case["codec"] == "scalar" else 16 if case["block_dim"] == 8 else 14)
    if case["codec"] == "scalar":
        E, E_inv = (m.to(rows.device).double() for m in _shaping(_basis()[0]))
        cents, bounds = (t.to(rows.device).double() for t in _scalar_tables(case["key_bits"]))
        for i in range(0, len(rows), step):
            r = rows[i:i + step]
            codes = torch.bucketize(_scalar_units(r) @ E.T, bounds)
            norm = r.double().norm(dim=-1, keepdim=True).to(r.dtype).double()
            out[i:i + step] = cents[codes] @ E_inv.T * norm
        return out.view(keys.shape)
    bd = case["block_dim"]
    E, _, cents, decoded = (t.to(rows.device).double() for t in _codebook(bd))
    ct = cents.transpose(1, 2).contiguous()
    for i in range(0, len(rows), step):
        r = rows[i:i + step].double().view(-1, D // bd, bd).transpose(0, 1).contiguous()
        x = torch.bmm(r, E.transpose(1, 2).contiguous())
        idx = (cents.square().sum(-1).unsqueeze(1) - 2 * torch.bmm(x, ct)).argmin(-1)
        hat = torch.gather(decoded, 1, idx.unsqueeze(-1).expand(-1, -1, bd))
        out[i:i + step] = hat.transpose(0, 1).reshape(-1, D)
    return out.view(keys.shape)


def _decoded_values(case, values):
    """What the value packer keeps of values [..., D]: min/max codes per group of
    32 with every step in the values' dtype, decoded in 64 bits."""
    g = values.reshape(-1, D // VALUE_GROUP, VALUE_GROUP)
    out = torch.empty(g.shape, dtype=torch.float64, device=g.device)
    # (a tensor: the quotient itself, where a number is multiplied by its inverse)
    top = torch.tensor(2 ** case["value_bits"] - 1, dtype=values.dtype, device=values.device)
    for i in range(0, len(g), 1 << 20):
        v = g[i:i + (1 << 20)]
        zero = v.amin(-1, keepdim=True)
        scale = ((v.amax(-1, keepdim=True) - zero) / top).clamp(min=1e-10)
        codes = torch.round((v - zero) / scale).clamp(0, 2 ** case["value_bits"] - 1)
        out[i:i + (1 << 20)] = codes.double() * scale.double() + zero.double()
    return out.view(values.shape)


def _attend(q, k, v, limit=None):
    """softmax(q k^T / sqrt(D)) v per KV head: q [T, Hq, D], k and v [N, Hkv, D]
    in 64 bits; key j is seen by query t if j <= limit[t]."""
    T, hq = q.shape[:2]
    h = k.shape[1]
    g = hq // h
    out = torch.empty(T, hq, D, dtype=torch.float64, device=q.device)
    for i in range(h):
        kt, vi = k[:, i].T.contiguous(), v[:, i].contiguous()
        for j in range(g):
            s = (q[:, i * g + j].double() @ kt) / math.sqrt(D)
            if limit is not None:
                s.masked_fill_(torch.arange(len(k), device=q.device) > limit.unsqueeze(1), -math.inf)
            out[:, i * g + j] = torch.softmax(s, dim=-1) @ vi
    return out


def exact(case, seed):
    kind = case["kind"]
    keys, values = _tokens_in(case, seed)
    if kind in ("encode", "append"):
        if kind == "append":
            keys, values = keys.transpose(0, 1), values.transpose(0, 1)
        zeros, tops = (torch.stack([f(v.reshape(*v.shape[:-1], -1, VALUE_GROUP), dim=-1).double() for v in values])
                       for f in (torch.amin, torch.amax))
        norms = torch.stack([k.double().norm(dim=-1) for k in keys]) if case["codec"] == "scalar" else None
        return {"codes": None, "norms": norms, "data": None, "scales": (tops - zeros) / (2 ** case["value_bits"] - 1),
                "zeros": zeros}
    if kind == "cache":
        q, n = _queries(case, (case["seqs"], case["kv_heads"], 1), seed), case["tokens"] - RING
        k = torch.cat([_decoded_keys(case, keys[:, :, :n].contiguous()), keys[:, :, n:].double()], 2)
        v = torch.cat([_decoded_values(case, values[:, :, :n].contiguous()), values[:, :, n:].double()], 2)
        scores = (k * q.double()).sum(-1).unsqueeze(2) / math.sqrt(D)
        return scores, torch.matmul(torch.softmax(scores, dim=-1), v)
    if kind == "step":
        rk, rv = _recent(case, seed)
        k, v = _decoded_keys(case, keys), _decoded_values(case, values)
        if rk is not None:
            k, v = torch.cat([k, rk.double()]), torch.cat([v, rv.double()])
        return _attend(_queries(case, (case["queries"], case["q_heads"]), seed), k, v, _positions(case))
    q = _queries(case, (case["seqs"], case["q_heads"]), seed)
    pairs = zip(keys, values) if kind == "batch" else zip(*(x.split(_lengths(case, seed)) for x in (keys, values)))
    return torch.stack([_attend(q[b:b + 1], _decoded_keys(case, k), _decoded_values(case, v))
                        for b, (k, v) in enumerate(pairs)])
