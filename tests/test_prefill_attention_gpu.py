"""Causal attention of prefill chunks on packed words (spk_prefill_attn) against
a float64 evaluation of the reference's composition (unpack-gather + softmax
with the offset causal mask, spikeinfer/attention.py:161-178, :320-330).

Outputs lie in [0, 1].  fp32: each weight is exact to 2**-23 and at most ~130
32-key sums are added per wave, so 4e-6; 16-bit outputs add half an ulp.
"""
from __future__ import annotations

import math

import pytest
import torch

from model_ref import gather_ref, pack_ref
from spikeinfer_amd import _lib, attention
from spikeinfer_amd.attention import AttentionMetadata, paged_attention
from spikeinfer_amd.kernels.spike_attention import paged_spike_attn_prefill

TOL = {torch.float32: 4e-6, torch.bfloat16: 4e-6 + 2.0**-9, torch.float16: 4e-6 + 2.0**-12}


def _case(T, Hq, Hkv, D, bs, chunks, seed, dev, q_density=0.25, density=0.25):
    """Packed q [T, n, Hq, W], caches, and per-chunk tables of shuffled blocks."""
    g = torch.Generator(device=dev).manual_seed(seed)
    spikes = lambda *s, p: pack_ref((torch.rand((*s, D), generator=g, device=dev) < p).float())
    n = sum(q for q, _ in chunks)
    need = [-(-(q + c) // bs) for q, c in chunks]
    blocks = sum(need) + 2
    k, v = (spikes(T, Hkv, blocks * bs, p=density) for _ in range(2))
    order = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed)).int()
    tables, rows, at, row = [], [], 0, 0
    for (q, _), nb in zip(chunks, need):
        tables.append(order[at:at + nb].to(dev))
        rows.append(row)
        at += nb
        row += q
    return spikes(T, n, Hq, p=q_density), k, v, tables, rows


def _want(qw, kd, vd, ctx, D):
    """float64 outputs [T, q_len, Hq, D] of one chunk from dense k, v [T, Hkv, S, D]."""
    bits = (qw.long()[..., None] >> torch.arange(32, device=qw.device)) & 1
    q = bits.flatten(-2)[..., :D].double().transpose(1, 2)  # [T, Hq, n, D]
    rep = q.shape[1] // kd.shape[1]
    k, v = kd.repeat_interleave(rep, 1), vd.repeat_interleave(rep, 1)
    s = q @ k.transpose(-1, -2) / math.sqrt(D)
    n, S = s.shape[-2:]
    s = s.masked_fill(torch.arange(S, device=q.device) > ctx + torch.arange(n, device=q.device)[:, None], -math.inf)
    return (torch.softmax(s, -1) @ v).transpose(1, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,Hq,Hkv,D,bs,chunks", [
    (4, 14, 2, 64, 16, [(1, 0), (5, 0), (33, 1)]),           # single rows, ragged row tiles
    (4, 14, 2, 64, 16, [(251, 0), (64, 4), (130, 1000)]),    # key tiles of all four waves
    (2, 14, 2, 64, 32, [(1200, 0)]),                         # four row tiles a workgroup
    (4, 14, 2, 64, 16, [(700, 333)]),                        # two
    (1, 4, 4, 32, 16, [(31, 0), (32, 32), (97, 31)]),        # one word, no GQA
    (2, 6, 2, 40, 16, [(50, 13)]),                           # channels past the head
    (2, 4, 1, 45, 16, [(20, 3)]),                            # rows without aligned stores
    (2, 6, 2, 96, 64, [(40, 70), (600, 0)]),
    (2, 16, 1, 128, 16, [(19, 5), (300, 129)]),
    (4, 8, 2, 128, 16, [(900, 0)]),
])
def test_matches_float64(gpu, T, Hq, Hkv, D, bs, chunks, dtype):
    q, k, v, tables, rows = _case(T, Hq, Hkv, D, bs, chunks, sum(map(sum, chunks)) + D, gpu)
    out = torch.full((T, q.shape[1], Hq, D), float("nan"), dtype=dtype, device=gpu)
    paged_spike_attn_prefill(q, k, v, [(r, r, n, c, t) for r, (n, c), t in zip(rows, chunks, tables)], out, D, bs)
    for r, (n, c), tab in zip(rows, chunks, tables):
        kd, vd = (gather_ref(x, tab, n + c, D, bs, torch.float64) for x in (k, v))
        want = _want(q[:, r:r + n], kd, vd, c, D)
        err = (out[:, r:r + n].double() - want).abs().max().item()
        assert err <= TOL[dtype], f"chunk {n}+{c}: {err}"


@pytest.mark.gpu
def test_dense_and_silent_words(gpu):
    """Densities 0 and 1: scores at both ends of the weight table, equal rows."""
    for D, Hq in ((64, 14), (128, 4)):
        for qd, kd_ in ((1.1, 1.1), (1.1, 0.0), (0.0, 1.1), (1.1, 0.5)):
            q, k, v, tables, _ = _case(2, Hq, 2, D, 16, [(70, 30)], 5, gpu, qd, kd_)
            out = torch.empty((2, 70, Hq, D), device=gpu)
            paged_spike_attn_prefill(q, k, v, [(0, 0, 70, 30, tables[0])], out, D, 16)
            kd, vd = (gather_ref(x, tables[0], 100, D, 16, torch.float64) for x in (k, v))
            assert (out.double() - _want(q, kd, vd, 30, D)).abs().max().item() <= TOL[torch.float32]


@pytest.mark.gpu
@pytest.mark.parametrize("density", [0.2, 0.5])
@pytest.mark.parametrize("D,Hq,Hkv", [(64, 14, 2), (32, 8, 8), (128, 8, 2), (96, 6, 2), (45, 6, 2)])
def test_fp32_outputs_keep_32_bits(gpu, D, Hq, Hkv, density):
    """fp32 outputs against float64 by the keys a row sees, and against the fp32
    composition (unpack-gather + SDPA).  The quotient is rounded once (at most 2**-24
    of the value, 3.4e-8 in the 2-norm); a weight is exact to 2**-23, and what its
    error leaves in a quotient of sums made of the same weights is below a third of
    that; sums of the weights' high halves are exact up to 2**24 of the smallest one's
    units.  So 4.5e-8 in the 2-norm, for short rows and long.  A row of one key is
    exact."""
    bits = lambda w: ((w.long()[..., None] >> torch.arange(32, device=gpu)) & 1).flatten(-2)[..., :D]
    for n, ctx, edges in ((300, 0, (1, 2, 4, 8, 16, 32, 64, 128, 300)), (64, 3900, (3964,)), (32, 12000, (12032,))):
        q, k, v, tables, _ = _case(2, Hq, Hkv, D, 16, [(n, ctx)], n + D, gpu, density, density)
        out, sdpa = (torch.empty((2, n, Hq, D), device=gpu) for _ in range(2))
        paged_spike_attn_prefill(q, k, v, [(0, 0, n, ctx, tables[0])], out, D, 16)
        meta = AttentionMetadata(slot_mapping=torch.arange(n, device=gpu), block_size=16, prefill_query_starts=[0],
                                 prefill_query_lens=[n], prefill_context_lens=[ctx], prefill_block_tables=tables)
        attention._prefill(bits(q).float().transpose(1, 2), k, v, meta, sdpa, Hq, Hkv, D)
        kd, vd = (gather_ref(x, tables[0], n + ctx, D, 16, torch.float64) for x in (k, v))
        want = _want(q, kd, vd, ctx, D)
        at = 0
        for edge in edges:
            rows = slice(at, edge - ctx)
            rel = [((o[:, rows].double() - want[:, rows]).norm() / want[:, rows].norm()).item() for o in (out, sdpa)]
            print(f"D={D} density={density} up to {edge} keys: {rel[0]:.2e}, sdpa {rel[1]:.2e}", flush=True)
            assert rel[0] <= (0.0 if edge == 1 else 4.5e-8), (edge, rel)
            at = edge - ctx


@pytest.mark.gpu
def test_contiguous_keys_short_tables_and_offsets(gpu):
    """Keys without a table (slot q_row + j), tables that end early or point
    outside the cache (zero spikes, still counted), a strided output at an
    offset from the query rows."""
    T, Hq, Hkv, D, bs = 4, 14, 2, 64, 16
    q, k, v, tables, _ = _case(T, Hq, Hkv, D, bs, [(90, 70)], 3, gpu)
    words = [x[:, :, :90].permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for x in (k, v)]
    big = torch.full((T, 200, Hq, D), -1.0, device=gpu)
    out = big[:, 60:]
    paged_spike_attn_prefill(q, *words, [(10, 17, 80, 0, None)], out, D, bs)
    bits = lambda x: ((x.long()[..., None] >> torch.arange(32, device=gpu)) & 1).flatten(-2).double()
    want = _want(q[:, 10:], bits(words[0])[:, :, 10:], bits(words[1])[:, :, 10:], 0, D)
    assert (out[:, 17:97].double() - want).abs().max().item() <= TOL[torch.float32]
    assert (big[:, :77] == -1).all() and (big[:, 157:] == -1).all()

    table = tables[0].clone()
    table[2], table[4] = 10**6, -1
    table = table[:7]  # 112 of the 160 tokens
    kd, vd = (gather_ref(x, tables[0], 160, D, bs, torch.float64) for x in (k, v))
    for d in (kd, vd):
        d[:, :, 32:48] = 0
        d[:, :, 64:80] = 0
        d[:, :, 112:] = 0
    o = torch.empty((T, 90, Hq, D), device=gpu)
    paged_spike_attn_prefill(q, k, v, [(0, 0, 90, 70, table.long())], o, D, bs)
    assert (o.double() - _want(q, kd, vd, 70, D)).abs().max().item() <= TOL[torch.float32]


@pytest.mark.gpu
def test_a_chunk_does_not_depend_on_its_batch(gpu):
    """Bit-identical alone, among 40 chunks (two launches) and beside one long
    enough to change the rows a workgroup takes."""
    T, Hq, Hkv, D, bs = 4, 14, 2, 64, 16
    chunks = [(37, 90)] + [(3 + i, 7 * i) for i in range(39)] + [(1500, 0)]
    q, k, v, tables, rows = _case(T, Hq, Hkv, D, bs, chunks, 9, gpu)
    args = [(r, r, n, c, t) for r, (n, c), t in zip(rows, chunks, tables)]
    outs = []
    for part in (args, args[:-1], args[:1]):
        out = torch.zeros((T, q.shape[1], Hq, D), device=gpu)
        paged_spike_attn_prefill(q, k, v, part, out, D, bs)
        outs.append(out[:, :37])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.gpu
def test_dense_query_gradients_and_wide_heads_keep_sdpa(gpu):
    """Dense queries that need gradients and head dims over 128 take the dense
    composition: gradients flow, values agree with the packed path."""
    T, n, bs = 2, 21, 16
    for D, grad in ((64, True), (160, False)):
        g = torch.Generator(device=gpu).manual_seed(D)
        spk = lambda h: (torch.rand((T, 1, h, n, D), generator=g, device=gpu) < 0.3).float()
        q, k, v = spk(4), spk(2), spk(2)
        caches = [torch.zeros((T, 2, 48, -(-D // 32)), dtype=torch.int32, device=gpu) for _ in range(2)]
        meta = AttentionMetadata(slot_mapping=torch.arange(n, device=gpu), block_size=bs, prefill_query_starts=[0],
                                 prefill_query_lens=[n], prefill_context_lens=[0],
                                 prefill_block_tables=[torch.arange(2, device=gpu, dtype=torch.int32)])
        out = paged_attention(q.requires_grad_(grad), k, v, *caches, meta, 4, 2, D)
        assert out.requires_grad == grad
        want = _want(pack_ref(q[:, 0].transpose(1, 2)), k[:, 0].double(), v[:, 0].double(), 0, D)
        assert (out.detach().view(T, n, 4, D).double() - want).abs().max().item() <= 1e-5
        if grad:
            out.sum().backward()
            assert q.grad is not None and torch.isfinite(q.grad).all()


def test_bad_chunks_are_refused_on_the_host():
    lib = _lib.load()
    s = (_lib.ctypes.c_int64 * 3)(1, 1, 1)
    call = lambda chunk, D=64, scale=0.125, dt=0, n=1: lib.spk_prefill_attn(
        16, s, 16, 16, s, 100, chunk, n, 16, dt, s, 4, 14, 2, D, 16, scale, None)
    ok = dict(start=0, table=0, table_stride=0, n_table=0, q_len=4, ctx=0)
    pack = lambda **k: _lib.pack_prefill_chunk(**{**ok, **k})
    assert call(pack(), D=160) == _lib.SPK_EUNSUPPORTED
    assert call(pack(), scale=0.5) == _lib.SPK_EINVAL
    assert call(pack(), dt=_lib.SPK_I32) == _lib.SPK_EINVAL
    assert call(pack(ctx=3)) == _lib.SPK_EINVAL       # cached prefix without a table
    assert call(pack(start=97)) == _lib.SPK_EINVAL    # past the slots
    assert call(pack(start=2**63 - 2)) == _lib.SPK_EINVAL  # (the end past 64 bits)
    assert call(pack(q_len=-1)) == _lib.SPK_EINVAL
    assert call(pack(), n=0) == _lib.SPK_OK
    assert call(pack(q_len=0)) == _lib.SPK_OK         # nothing to do, nothing launched
    assert len(pack()) == 40
