"""The matrix-core row kernel (attention_rows.h: block-VQ keys, more than 4
query rows per KV head, 4-bit values) against the generic kernels (impl 1,
oracle-checked in test_gpu_attention.py), at its tile and share edges.

Outputs are fp32.  Either side's logits are within 2^-22 * sum |q k| * scale of
the exact ones (at most 40 here: 1e-5), its weights within as much relative,
and the weights sum to 1, so outputs agree to 2e-5 * max |v|."""

from __future__ import annotations

import pytest
import torch

import smaq_amd as S
from smaq_amd.batch import PagedQuantizedKV, QuantizedKVBatch
from smaq_amd.score import plan_hybrid_attention
from tests.conftest import sample_keys

pytestmark = pytest.mark.gpu


def _strategy(dev, codec, size, seed=0):
    if codec == "scalar":
        return S.SMAQFullMetricScalarStrategy(128, bits=size, device=dev).fit(sample_keys(64, seed=seed + 5))
    nc = 100 if size == 4 else 256
    strat = S.SMAQBlockVQStrategy(128, block_dim=size, n_centroids=nc, device=dev)
    x = sample_keys(nc, seed=seed + 6).reshape(nc, 128 // size, size).transpose(0, 1).contiguous().to(dev)
    strat.quantizer.load_state_dict({**strat.quantizer.state_dict(), "centroids": x, "decoded_centroids": x})
    return strat


def _takes_rows(plan, q, got):
    """Whether ``got`` is the row kernel's: without arrival counters the same
    plan runs the kernels it would otherwise run, whose bits repeat."""
    arrivals, plan.params.arrivals = plan.params.arrivals, None
    other = plan.run(q).view_as(got).clone()
    again = torch.equal(plan.run(q).view_as(got), other)
    plan.params.arrivals = arrivals
    return again and not torch.equal(other, got)


def _close(got, ref, vals, what):
    diff = float((got - ref).abs().max())
    print(f"\n[{what}] max|err| {diff:.2e}")
    assert diff <= 2e-5 * float(max(v.float().abs().max() for v in vals)), what


# (codec, key bits or block dim, value bits, heads per KV head, query tokens, storage dtype)
FORMS = [("vq", 2, 2, 7, 1, torch.float16), ("vq", 4, 4, 8, 1, torch.bfloat16), ("vq", 8, 2, 4, 3, torch.bfloat16),
         ("vq", 8, 4, 1, 1, torch.float32), ("scalar", 3, 2, 7, 1, torch.bfloat16), ("scalar", 4, 4, 3, 1, torch.float16),
         ("scalar", 3, 4, 2, 15, torch.float32), ("scalar", 4, 2, 16, 2, torch.float32), ("vq", 2, 4, 3, 63, torch.bfloat16)]


@pytest.mark.parametrize("codec,size,vbits,g,T,dtype", FORMS)
def test_rows_store_edges(dev, codec, size, vbits, g, T, dtype):
    """One sequence, lengths around the 32-token tile, the steps of 128 and 256
    tokens and a share of several steps; with and without a recent window and
    a causal limit; a repeated call gives the same bits."""
    strat = _strategy(dev, codec, size)
    for n, rn in ((63, 0) if T > 16 else (16, 0), (33, 31) if T > 16 else (33, 1), (127, 64), (257, 65), (513, 0), (2051, 128)):
        st = S.CompressedKVStore(128, 2, value_bits=vbits, device=dev, key_strategy=strat)
        k = sample_keys(n * 2, seed=n).view(n, 2, 128).to(dtype).to(dev)
        v = torch.randn(n, 2, 128, generator=torch.Generator().manual_seed(n)).to(dtype).to(dev)
        st.append_chunk(k, v)
        q = sample_keys(T * 2 * g, seed=n + 1).view(T, 2 * g, 128).to(dev)
        kr = sample_keys(max(rn, 1) * 2, seed=n + 2).view(-1, 2, 128).to(dtype).to(dev) if rn else None
        pos = torch.arange(n + rn - T, n + rn, device=dev) if T > 1 else None
        got = S.compute_hybrid_attention(q, st, kr, kr, 2 * g, query_positions=pos)
        ref = S.compute_hybrid_attention(q, st, kr, kr, 2 * g, query_positions=pos, impl=1)
        _close(got, ref, (v,) if kr is None else (v, kr), f"{codec}{size} v{vbits} g{g} T{T} n{n} r{rn}")
        again = S.compute_hybrid_attention(q, st, kr, kr, 2 * g, query_positions=pos)
        assert torch.equal(got, again)
        assert _takes_rows(plan_hybrid_attention(q, st, kr, kr, 2 * g, query_positions=pos), q.unsqueeze(0), got), (n, rn)


@pytest.mark.parametrize("codec,size,vbits,g,T,dtype", FORMS[:7:3] + FORMS[4:5])
@pytest.mark.parametrize("block_size", [0, 16, 64])
def test_rows_ragged_batches(dev, codec, size, vbits, g, T, dtype, block_size):
    """Ragged sequences (odd first rows, more than the 64 of one scan step),
    contiguous or in shuffled pages, then shorter lengths set on the same plan:
    zero, one token, a part of a page.  The counters are left at zero."""
    strat = _strategy(dev, codec, size, seed=9)
    lens = [(37 * i * i) % 389 + 1 for i in range(66)] + [1500]
    gen = torch.Generator().manual_seed(3)
    keys = [sample_keys(n * 2, seed=i).view(n, 2, 128).to(dtype).to(dev) for i, n in enumerate(lens)]
    vals = [torch.randn(n, 2, 128, generator=gen).to(dtype).to(dev) for n in lens]
    # (N(0, 1) queries reach logits of 366 in the calibrated metric, where either
    # side is 1.2e-4 off the float64 result: 2^-22 * 366 = 9e-5, times |v|)
    q = sample_keys(len(lens) * T * 2 * g, seed=99).view(len(lens), T, 2 * g, 128).to(dev)
    if block_size:
        need = [-(-n // block_size) for n in lens]
        perm = torch.randperm(sum(need), generator=gen).to(torch.int32)
        table = torch.zeros(len(lens), max(need), dtype=torch.int32)
        for i, (c, part) in enumerate(zip(need, perm.split(need))):
            table[i, :c] = part
        kv = PagedQuantizedKV.encode(strat, keys, vals, table.to(dev), sum(need), block_size=block_size, value_bits=vbits)
    else:
        kv = QuantizedKVBatch.encode(strat, keys, vals, value_bits=vbits)
    plans = [kv.plan(q, impl=i) for i in (0, 1)]
    for cut in (None, torch.tensor([(n * i) % (n + 1) for i, n in enumerate(lens)])):
        for p in plans:
            if cut is not None:
                p.set_lengths(hist_len=cut)
        got, ref = (p.run(q).clone() for p in plans)
        _close(got, ref, vals, f"{codec}{size} v{vbits} g{g} T{T} block {block_size} {'cut' if cut is not None else ''}")
        assert _takes_rows(plans[0], q, got)
        assert not plans[0].arrivals.any()


def test_rows_value_scale_range_and_nan(dev):
    """Value scales from 2^-24 to 2^15 across tokens (the weights' exponent
    follows the largest), then a NaN key norm: its row's outputs are NaN."""
    strat = _strategy(dev, "scalar", 3)
    n, g = 700, 8
    v = torch.randn(n, 2, 128, generator=torch.Generator().manual_seed(1))
    v[100:200] *= 2.0 ** -24
    v[300:310] *= 2.0 ** 15
    k = sample_keys(n * 2, seed=2).view(n, 2, 128)
    kv = QuantizedKVBatch.encode(strat, [k.to(dev)], [v.to(dev)])
    q = sample_keys(2 * g, seed=3).view(1, 2 * g, 128).to(dev)
    got, ref = kv.attention(q), kv.attention(q, impl=1)
    _close(got, ref, (v,), "scales")
    kv.norms[1, 350] = float("nan")
    bad = kv.attention(q)
    assert bool(bad[:, g:].isnan().all()) and torch.equal(bad[:, :g], got[:, :g])


def test_rows_small_workspace_runs_generic(dev):
    """A workspace of the generic kernels' size (sized without arrival
    counters) is still enough."""
    import ctypes
    from smaq_amd import _native
    strat = _strategy(dev, "vq", 8)
    n = 400
    k = sample_keys(n * 2, seed=5).view(n, 2, 128).to(dev)
    kv = QuantizedKVBatch.encode(strat, [k], [k])
    q = sample_keys(4, seed=6).view(1, 4, 128).to(dev)
    plan = kv.plan(q)
    want = kv.attention(q, impl=1)
    arrivals, plan.params.arrivals = plan.params.arrivals, None
    small = _native.lib().smaq_attn_workspace_bytes(ctypes.byref(plan.params))
    plan.params.arrivals = arrivals
    assert small < plan.params.workspace_bytes
    plan.params.workspace_bytes = small
    assert torch.equal(plan.run(q).view_as(want), want)


@pytest.mark.parametrize("T,rn,impl,dtype", [(1, 0, 0, torch.bfloat16), (1, 70, 0, torch.float16), (3, 129, 0, torch.bfloat16),
                                             (63, 5, 0, torch.float32), (1, 70, 1, torch.bfloat16),
                                             (64, 40, 3, torch.bfloat16), (64, 0, 0, torch.float16)])
def test_unrotated_query_is_widened_by_the_library(dev, T, rn, impl, dtype):
    """A run of an unrotated codec's plan gives the bits of a loaded query and
    a launch, leaves the fp32 query in q_exact for a later launch, and keeps
    no pointer to the caller's query; a strided query still runs."""
    n, g = 300, 3
    k = sample_keys(2 * n * 2, seed=1).view(2, n, 2, 128).to(dev)
    v = torch.randn(2, n, 2, 128, generator=torch.Generator().manual_seed(2)).to(dev)
    kvb = QuantizedKVBatch.encode(_strategy(dev, "vq", 8), k, v)
    q = sample_keys(2 * T * 2 * g, seed=3).view(2, T, 2 * g, 128).to(dtype).to(dev)
    rk = sample_keys(2 * rn * 2, seed=4).view(2, rn, 2, 128).bfloat16().to(dev) if rn else None
    plan = kvb.plan(q, None, rk, rk, torch.tensor([0, rn], device=dev) if rn else None, impl)
    plan.load_query(q)
    ref = plan.launch().clone()
    plan.q_exact.fill_(float("nan"))
    assert torch.equal(plan.run(q), ref) and torch.equal(plan.q_exact, q.float())
    assert plan.params.q_raw is None and plan.params.phases == 0
    assert torch.equal(plan.launch(), ref)
    strided = torch.stack([q, q + 1], dim=-1)[..., 0]
    plan.q_exact.fill_(float("nan"))
    assert torch.equal(plan.run_into(strided, torch.empty_like(plan.out)), ref)
    plan.q_exact.fill_(float("nan"))
    assert torch.equal(plan.run_into(q, torch.empty_like(plan.out)), ref)


@pytest.mark.parametrize("scale", [0.0, -0.05, 1e-42])
@pytest.mark.parametrize("codec,size,vbits,g,T,dtype", [FORMS[0], FORMS[3], FORMS[4], FORMS[6]])
def test_rows_any_scale(dev, codec, size, vbits, g, T, dtype, scale):
    """A score scale that is zero, negative or below fp32's normal range:
    tokens past the length or the causal limit stay masked."""
    strat = _strategy(dev, codec, size)
    for n, rn in ((77, 0), (300, 9)):
        st = S.CompressedKVStore(128, 2, value_bits=vbits, device=dev, key_strategy=strat)
        k = sample_keys(n * 2, seed=n).view(n, 2, 128).to(dtype).to(dev)
        v = torch.randn(n, 2, 128, generator=torch.Generator().manual_seed(n)).to(dtype).to(dev)
        st.append_chunk(k, v)
        q = sample_keys(T * 2 * g, seed=n + 1).view(T, 2 * g, 128).to(dev)
        kr = sample_keys(max(rn, 1) * 2, seed=n + 2).view(-1, 2, 128).to(dtype).to(dev) if rn else None
        pos = torch.arange(n + rn - T, n + rn, device=dev) if T > 1 else None
        got, ref = (S.compute_hybrid_attention(q, st, kr, kr, 2 * g, scale=scale, query_positions=pos, impl=i) for i in (0, 1))
        _close(got, ref, (v,) if kr is None else (v, kr), f"{codec}{size} g{g} T{T} n{n} r{rn} scale {scale}")


@pytest.mark.parametrize("how", ["channel 1e4", "channel 1e6", "channel 1e9", "one value 1e9", "infinite scale",
                                 "token of little weight 1e6", "zero up to a late token"])
@pytest.mark.parametrize("codec,size,vbits,g,dtype", [("vq", 8, 2, 8, torch.bfloat16), ("scalar", 3, 4, 7, torch.float32)])
def test_rows_value_groups_far_apart(dev, codec, size, vbits, g, dtype, how):
    """Each group of 32 value dims is as exact as when it stands alone: one
    group's scales far above the others', at every token, at one, infinite, at
    a token of next to no weight, or zero up to a late token.  Tolerance: the
    file's, of the largest value of the group itself (the light token's left
    out)."""
    strat = _strategy(dev, codec, size)
    n, gen = 1500, torch.Generator().manual_seed(8)
    k = sample_keys(n * 2, seed=5).view(n, 2, 128).to(dtype).to(dev)
    v = torch.randn(n, 2, 128, generator=gen)
    q = 60 * sample_keys(2 * g, seed=6).view(1, 2 * g, 128).to(dev)   # (logits up to 30)
    live = torch.ones(n, 2, dtype=torch.bool)
    if how.startswith("channel"):
        v[:, :, 7] *= float(how.split()[1])
    elif how == "one value 1e9":
        v[700, 1, 40] = 1e9
    elif how == "token of little weight 1e6":
        khat = strat.dequantize(strat.quantize(k)).float().cpu()
        logits = torch.einsum("nhd,hgd->nhg", khat, q.cpu().view(2, g, 128)) * 128 ** -0.5
        light = torch.softmax(logits, 0).amax(2).argmin(0)
        for h in range(2):
            v[light[h], h] *= 1e6
            live[light[h], h] = False
    elif how == "zero up to a late token":
        v[:1300, :, 64:96] = 0.0
    v = v.to(dtype).to(dev)
    kv = QuantizedKVBatch.encode(strat, [k], [v], value_bits=vbits)
    if how == "infinite scale":
        kv.v_scales[1, 700, 2] = float("inf")
    got, ref = kv.attention(q), kv.attention(q, impl=1)
    top = (v.float() * live.to(dev).unsqueeze(-1)).view(n, 2, 4, 32).abs().amax((0, 3))   # [Hkv, group]
    err = (got - ref).view(2, g, 4, 32).abs().amax((1, 3))
    for h in range(2):
        for i in range(4):
            if how == "infinite scale" and (h, i) == (1, 2):
                assert not got.view(2, g, 4, 32)[h, :, i].isfinite().any()
                continue
            print(f"\n[{codec}{size} {how} head {h} group {i}] max|err| {float(err[h, i]):.2e} of {float(top[h, i]):.2e}")
            assert float(err[h, i]) <= 2e-5 * float(top[h, i])


@pytest.mark.parametrize("what", ["queries 2^-118", "queries 2^-130", "codebook 2^-118", "one block 2^40", "one block 2^-40"])
@pytest.mark.parametrize("size", [2, 4, 8])
def test_rows_query_and_codebook_range(dev, size, what):
    """Queries and codebooks at the edge of fp32's range (the score scale makes
    up for it), and a block whose codewords are far larger or smaller than the
    others' with its query dims the inverse: every block counts alike."""
    strat = _strategy(dev, "vq", size)
    n, g, nb = 333, 4, 128 // size
    k = sample_keys(n * 2, seed=5).view(n, 2, 128)
    v = torch.randn(n, 2, 128, generator=torch.Generator().manual_seed(4))
    kv = QuantizedKVBatch.encode(strat, [k.to(dev)], [v.to(dev)])
    q = sample_keys(2 * g, seed=6).view(1, 2 * g, 128).to(dev)
    scale, power = 128 ** -0.5, what.split("2^")[1]
    f = 2.0 ** int(power)
    state = strat.quantizer.state_dict()
    C = state["decoded_centroids"].clone()
    if what.startswith("queries"):
        q, scale = q * f, scale * 2.0 ** min(-int(power), 126)
    elif what.startswith("codebook"):
        C, scale = C * f, scale / f
    else:
        C[nb // 2] *= f
        q.view(1, 2 * g, nb, size)[:, :, nb // 2] /= f
    strat.quantizer.load_state_dict({**state, "decoded_centroids": C})
    got, ref = (kv.attention(q, scale=scale, impl=i) for i in (0, 1))
    assert float((ref - ref.mean(1, keepdim=True)).abs().max()) > 1e-3
    _close(got, ref, (v,), f"vq{size} {what}")


@pytest.mark.parametrize("codec,size,vbits,g,T,dtype", [FORMS[0], FORMS[4], FORMS[6]])
@pytest.mark.parametrize("rn", [0, 70])
def test_rows_shapes_in_separate_phases(dev, codec, size, vbits, g, T, dtype, rn):
    """Phases launched apart, whichever are joined, give the generic kernels'
    result."""
    strat = _strategy(dev, codec, size)
    n = 400
    k = sample_keys(2 * n * 2, seed=1).view(2, n, 2, 128).to(dtype).to(dev)
    v = torch.randn(2, n, 2, 128, generator=torch.Generator().manual_seed(2)).to(dtype).to(dev)
    kv = QuantizedKVBatch.encode(strat, k, v, value_bits=vbits)
    q = sample_keys(2 * T * 2 * g, seed=3).view(2, T, 2 * g, 128).to(dev)
    rk = sample_keys(2 * rn * 2, seed=4).view(2, rn, 2, 128).to(dtype).to(dev) if rn else None
    rl = torch.tensor([rn, rn // 2], device=dev) if rn else None
    ref = kv.plan(q, None, rk, rk, rl, impl=1).run(q)
    plan = kv.plan(q, None, rk, rk, rl)
    vals = (v,) if rk is None else (v, rk)
    _close(plan.run(q), ref, vals, "one call")
    for masks in ((8, 1, 2, 4), (8 | 1 | 2, 4), (8, 1, 2 | 4), (8 | 2, 1 | 4), (8, 1 | 2 | 4)):
        plan.load_query(q)
        plan.out.fill_(float("nan"))
        for m in masks:
            plan.launch(m)
        _close(plan.out, ref, vals, f"{codec}{size} T{T} r{rn} phases {masks}")


def test_rows_past_the_built_in_scratch(dev):
    """A batch whose row-kernel workspace passes the allocation-free entry
    point's scratch: a plan owns its workspace and takes the row kernel; the
    allocation-free call, whose generic workspace fits, still runs."""
    import ctypes
    from smaq_amd import _native
    strat = _strategy(dev, "vq", 8)
    B, H, n, g = 700, 16, 40, 1
    k = sample_keys(n * H, seed=1).view(1, n, H, 128).to(dev) + 0.1 * torch.randn(
        B, 1, H, 1, generator=torch.Generator().manual_seed(3)).to(dev)
    kv = QuantizedKVBatch.encode(strat, k, k)
    q = sample_keys(B * H * g, seed=2).view(B, H * g, 128).to(dev)
    plan = kv.plan(q)
    generic = kv.plan(q, impl=1).params.workspace_bytes
    slots = B * H * 8 * 130 * 4
    assert generic < _native.NOALLOC_SCRATCH_BYTES < slots
    assert plan.params.workspace_bytes > slots
    got, ref = plan.run(q).clone(), kv.attention(q, impl=1).view_as(plan.out)
    _close(got, ref, (k,), "700 x 16 units")
    assert not torch.equal(got, ref)       # (the row kernel's sums, not the generic one's)
    plan.load_query(q)
    plan.out.fill_(float("nan"))
    _native.attn_hybrid_noalloc(plan.params, dev)
    assert torch.equal(plan.out, ref)


@pytest.mark.parametrize("codec,size", [("vq", 8), ("scalar", 3)])
@pytest.mark.parametrize("T,n,rn,prefill,dtype", [(63, 500, 4096, True, torch.bfloat16), (63, 500, 128, False, torch.bfloat16),
                                                  (63, 30000, 4096, False, torch.bfloat16), (16, 500, 4096, False, torch.bfloat16),
                                                  (32, 500, 16384, True, torch.bfloat16), (63, 500, 4096, False, torch.float32),
                                                  (63, 500, 4096, False, torch.float16)])
def test_rows_long_window_chunks(dev, codec, size, T, n, rn, prefill, dtype):
    """Chunks beside a long exact window: the window's cost counts in the
    choice between the row and the prefill kernel, where the latter is as exact."""
    strat = _strategy(dev, codec, size)
    st = S.CompressedKVStore(128, 4, device=dev, key_strategy=strat)
    k = sample_keys(n * 4, seed=n).view(n, 4, 128).to(dtype).to(dev)
    st.append_chunk(k, k)
    q = sample_keys(T * 28, seed=T).view(T, 28, 128).to(dev)
    kr = sample_keys(rn * 4, seed=rn).view(rn, 4, 128).to(dtype).to(dev)
    pos = torch.arange(n + rn - T, n + rn, device=dev)
    got, big, ref = (S.compute_hybrid_attention(q, st, kr, kr, 28, query_positions=pos, impl=i) for i in (0, 3, 1))
    assert torch.equal(got, big) == prefill
    _close(got, ref, (k, kr), f"{codec}{size} T{T} n{n} r{rn} {dtype}")


@pytest.mark.parametrize("size,B,n,T,hq,h,rn,rows", [(8, 512, 16, 3, 32, 8, 0, False), (8, 512, 100, 3, 32, 8, 0, True),
                                                      (8, 512, 16, 3, 8, 8, 0, True), (8, 200, 16, 3, 8, 8, 32, False),
                                                      (2, 200, 16, 24, 28, 4, 0, False), (2, 200, 1000, 24, 28, 4, 0, True)])
def test_rows_many_short_sequences(dev, size, B, n, T, hq, h, rn, rows):
    """Many sequences of a few tokens, whose units the generic and prefill kernels
    work through faster: without arrival counters, which the row kernel needs,
    the same call gives the same bits where it did not run."""
    strat = _strategy(dev, "vq", size)
    k = sample_keys(B * n * h, seed=1).view(B, n, h, 128).bfloat16().to(dev)
    kv = QuantizedKVBatch.encode(strat, k, k)
    q = sample_keys(B * T * hq, seed=2).view(B, T, hq, 128).to(dev)
    rk = sample_keys(B * rn * h, seed=3).view(B, rn, h, 128).bfloat16().to(dev) if rn else None
    plan = kv.plan(q, None, rk, rk)
    got = plan.run(q).clone()
    _close(got, kv.plan(q, None, rk, rk, impl=1).run(q), (k,), f"vq{size} B{B} n{n} T{T} r{rn}")
    assert _takes_rows(plan, q, got) == rows


@pytest.mark.parametrize("codec,size", [("scalar", 3), ("vq", 2), ("vq", 8)])
@pytest.mark.parametrize("n", [1, 31, 128, 129, 257, 513])
def test_rows_shares_of_whole_units(dev, codec, size, n):
    """Histories below the least share: a unit a share, whole; above it, in
    pieces; lengths that differ included."""
    strat = _strategy(dev, codec, size)
    B, h, g, T = 5, 2, 2, 7
    k = sample_keys(B * n * h, seed=1).view(B, n, h, 128).to(dev)
    kv = QuantizedKVBatch.encode(strat, k, k)
    q = sample_keys(B * T * h * g, seed=2).view(B, T, h * g, 128).to(dev)
    plans = [kv.plan(q, impl=i) for i in (0, 1)]
    for cut in (None, [n, 0, 1, max(n - 1, 0), n // 2]):
        if cut is not None and plans[0].hist_len is None:
            continue
        for p in plans:
            if cut is not None:
                p.set_lengths(hist_len=torch.tensor(cut, device=dev))
        got, ref = (p.run(q).clone() for p in plans)
        _close(got, ref, (k,), f"{codec}{size} n{n} {cut}")
        assert torch.equal(got, plans[0].run(q))
