"""Which form of the prefill attention a call takes, and what it does with the
forms of its arguments, on the CPU: the kernels' wrappers are replaced by plain
torch, the packed kernel by a float64 evaluation of its words."""
from __future__ import annotations

import math

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.nn.attention import SDPBackend, sdpa_kernel

import spikeinfer_amd.attention as A
from model_ref import gather_ref, lif_ref, pack_ref, unpack_ref
from spikeinfer_amd.attention import AttentionMetadata, paged_attention, paged_attention_fused
from spikeinfer_amd.kernels.spike_attention import PREFILL_DTYPES

T, HQ, HKV, D, BS = 2, 4, 2, 64, 16


@pytest.fixture
def packed_calls(monkeypatch):
    """Plain torch in the kernels' place; the calls of the packed prefill kernel."""
    calls = []

    def prefill(q, k, v, chunks, out, head_dim, block_size):
        # what the kernel's wrapper asks of them
        assert out.stride(-1) == 1 and out.dtype in PREFILL_DTYPES
        calls.append(chunks)
        for q_row, out_row, n, ctx, table in chunks:
            kd, vd = (gather_ref(c, table, ctx + n, head_dim, block_size, torch.float64) for c in (k, v))
            qd = unpack_ref(q[:, q_row:q_row + n], head_dim, torch.float64).transpose(1, 2)
            rep = qd.shape[1] // kd.shape[1]
            s = qd @ kd.repeat_interleave(rep, 1).transpose(-1, -2) / math.sqrt(head_dim)
            s = s.masked_fill(torch.arange(ctx + n) > ctx + torch.arange(n)[:, None], -math.inf)
            out[:, out_row:out_row + n] = (torch.softmax(s, -1) @ vd.repeat_interleave(rep, 1)).transpose(1, 2)
        return out

    def sites(every, slots=None):
        assert len({x.dtype for x, *_ in every}) == 1  # what the kernel's wrapper asks
        for x, beta, th, out, scatter in every:
            words = pack_ref(lif_ref(x, beta, th))
            out.index_copy_(2, slots, words.transpose(1, 2)) if scatter else out.copy_(words)

    def pack(x):
        x.data_ptr()  # (raises for a tensor without storage, as the kernel's wrapper does)
        return pack_ref(x)

    monkeypatch.setattr(A, "pack_spikes", pack)
    monkeypatch.setattr(A, "gather_kv_unpacked_pair",
                        lambda k, v, *a: (gather_ref(k, *a), gather_ref(v, *a)))
    monkeypatch.setattr(A, "paged_spike_attn_prefill", prefill)
    monkeypatch.setattr(A, "lif_pack_write_sites", sites)
    return calls


def _spikes(n, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [(torch.rand((T, 1, h, n, D), generator=g) < 0.3).float() for h in (HQ, HKV, HKV)]


def _meta(lens, ctx=None, tables=None):
    n, starts = sum(lens), [sum(lens[:i]) for i in range(len(lens))]
    tables = tables if tables is not None else [torch.arange(4 * i, 4 * i + 4).int() for i in range(len(lens))]
    slots = torch.cat([4 * BS * i + torch.arange(m) for i, m in enumerate(lens)])
    return AttentionMetadata(slot_mapping=slots, block_size=BS, prefill_query_starts=starts, prefill_query_lens=lens,
                             prefill_context_lens=ctx or [0] * len(lens), prefill_block_tables=tables)


def _caches():
    return [torch.zeros((T, HKV, 12 * BS, 2), dtype=torch.int32) for _ in range(2)]


def _attend(n):
    """The step as a function of its queries."""
    (_, k, v), caches, meta = _spikes(n), _caches(), _meta([n])
    return lambda q: paged_attention(q, k, v, *caches, meta, HQ, HKV, D)


def test_plain_queries_take_the_packed_kernel(packed_calls):
    q, attend = _spikes(9)[0], _attend(9)
    plain = attend(q)
    with torch.no_grad():
        off = attend(q.clone().requires_grad_())
    assert len(packed_calls) == 2 and torch.equal(plain, off)
    grad = attend(q.clone().requires_grad_())
    assert len(packed_calls) == 2 and grad.requires_grad
    torch.testing.assert_close(grad.detach(), plain, rtol=0, atol=1e-6)


def test_derivatives_to_the_queries_flow_in_every_mode(packed_calls):
    """Reverse and forward mode: neither may end in packed words.  (torch.func's
    transforms wrap the k spikes too, which the packing refuses.)"""
    q, attend = _spikes(9)[0], _attend(9)
    d = torch.randn(q.shape, generator=torch.Generator().manual_seed(1))
    leaf = q.clone().requires_grad_()
    with sdpa_kernel(SDPBackend.MATH):  # (the only backend with a forward mode)
        reverse = torch.autograd.grad(attend(leaf).square().sum(), leaf)[0]
        with fwAD.dual_level():
            out = fwAD.unpack_dual(attend(fwAD.make_dual(q, d)))
            assert out.tangent is not None
            forward = (2 * out.primal * out.tangent).sum()
        with pytest.raises(RuntimeError, match="storage"):
            torch.func.grad(lambda x: attend(x).sum())(q)
    torch.testing.assert_close(forward, (reverse * d).sum(), rtol=1e-4, atol=1e-4)
    assert not packed_calls
    with fwAD.dual_level():  # a level without a tangent to the queries
        attend(q)
    assert len(packed_calls) == 1


def test_every_chunk_needs_its_entry_in_each_list(packed_calls):
    """A list shorter than the chunks' lengths is an error, not rows left unwritten;
    entries past them are not looked at."""
    q, k, v = _spikes(12)
    run = lambda meta: paged_attention(q, k, v, *_caches(), meta, HQ, HKV, D)
    good = run(_meta([5, 7]))
    for name in ("prefill_query_starts", "prefill_context_lens", "prefill_block_tables"):
        meta = _meta([5, 7])
        setattr(meta, name, getattr(meta, name)[:1])
        with pytest.raises(IndexError):
            run(meta)
        meta = _meta([5, 7])
        setattr(meta, name, getattr(meta, name) * 2)
        assert torch.equal(run(meta), good)


def _fused(n, out=None, q_dtype=torch.float32, **over):
    g = torch.Generator().manual_seed(n)
    cur = [torch.randn((T, n, h, D), generator=g) for h in (HQ, HKV, HKV)]
    cur[0] = cur[0].bfloat16().to(q_dtype)
    lif = [(torch.full((D,), 0.9), torch.full((D,), 1.0))] * 3
    return paged_attention_fused(*cur, *lif, *_caches(), _meta([5, n - 5]), HQ, HKV, D, out=out)


def test_fused_outputs_of_any_type_and_layout(packed_calls):
    """The kernel writes floats with contiguous channels; other `out` tensors
    receive the chunks' rows too, and nothing else of them is touched."""
    n = 12
    want = _fused(n)
    for dtype, step in ((torch.float64, 1), (torch.float32, 2), (torch.bfloat16, 2)):
        big = torch.full((T, n + 2, HQ, step * D), -7.0, dtype=dtype)
        out = big[:, :n, :, ::step]
        got = _fused(n, out)
        assert got.dtype == dtype and got.data_ptr() == big.data_ptr()
        assert torch.equal(got, want.to(dtype))
        assert (big[:, n:] == -7).all() and (step == 1 or (big[:, :, :, 1::step] == -7).all())


def test_fused_query_currents_of_their_own_type(packed_calls):
    """Query currents in another float type than k and v (one launch takes one type)."""
    want = _fused(12)
    got = _fused(12, q_dtype=torch.bfloat16)
    assert got.dtype == torch.bfloat16 and torch.equal(got, want.bfloat16())


@pytest.mark.parametrize("lens,ctx", [([20, 20, 20], [0, 0, 0]), ([20, 33, 1], [0, 0, 0]),
                                      ([7, 20, 20], [40, 0, 0]), ([9, 5], [33, 20])])
def test_dense_prefill_of_wide_heads(monkeypatch, lens, ctx):
    """SpikingDecoder's dense form, which heads of more than 128 channels take: fresh
    chunks of one length in one batched call, ragged ones, and cached prefixes."""
    import spikeinfer_amd.model as M

    D, n = 256, sum(lens)
    g = torch.Generator().manual_seed(n)
    monkeypatch.setattr(M, "gather_kv_unpacked_pair", lambda k, v, *a: (gather_ref(k, *a), gather_ref(v, *a)))
    caches = [pack_ref((torch.rand((T, HKV, 12 * BS, D), generator=g) < 0.3).float()) for _ in range(2)]
    dense = [(torch.rand((T, h, n, D), generator=g) < 0.3).float() for h in (HQ, HKV, HKV)]
    meta = _meta(lens, ctx)
    for i, (start, m, c) in enumerate(zip(meta.prefill_query_starts, lens, ctx)):  # the chunk's own k and v
        for cache, d in zip(caches, dense[1:]):
            cache[:, :, 4 * BS * i + c:4 * BS * i + c + m] = pack_ref(d[:, :, start:start + m])
    model = M.SpikingDecoder.__new__(M.SpikingDecoder)
    model.T, model.D, model.Hq, model.Hkv, model.dtype = T, D, HQ, HKV, torch.float32
    attn = torch.full((T, n, HQ, D), float("nan"))
    model._prefill_attention(dense, *caches, meta, attn)
    for i, (start, m, c) in enumerate(zip(meta.prefill_query_starts, lens, ctx)):
        k, v = (gather_ref(x, meta.prefill_block_tables[i], c + m, D, BS, torch.float64) for x in caches)
        q = dense[0][:, :, start:start + m].double()
        s = q @ k.repeat_interleave(HQ // HKV, 1).transpose(-1, -2) / math.sqrt(D)
        s = s.masked_fill(torch.arange(c + m) > c + torch.arange(m)[:, None], -math.inf)
        want = (torch.softmax(s, -1) @ v.repeat_interleave(HQ // HKV, 1)).transpose(1, 2)
        # (values in [0, 1], at most 49 fp32 terms: 49 * 2**-24)
        torch.testing.assert_close(attn[:, start:start + m].double(), want, rtol=0, atol=3e-6)
