"""The C++ entry of the launch-bound operators (csrc/native.cpp) against the
wrappers' own path: same outputs, and calls it does not take (other dtypes,
strides, CPU tensors, wrong shapes) end as they do without it."""
from __future__ import annotations

import contextlib

import pytest
import torch

from spikeinfer_amd import _lib
from spikeinfer_amd.kernels import (lif_multistep, lif_pack_write_sites, pack_spikes, paged_spike_attn_decode)
from spikeinfer_amd.kernels.spike_attention import paged_spike_attn_prefill

pytestmark = pytest.mark.gpu
T, N, HQ, HKV, BS = 4, 5, 14, 2, 16


@contextlib.contextmanager
def _without_native():
    was, _lib._native = _lib.native(), None
    try:
        yield
    finally:
        _lib._native = was


def _inputs(gpu, D=64):
    g = torch.Generator(device=gpu).manual_seed(D)
    bits = lambda *s: pack_spikes(torch.rand((*s, D), generator=g, device=gpu) < 0.3)
    slots = N * 4 * BS
    return dict(q=bits(T, N, HQ), k=bits(T, HKV, slots), v=bits(T, HKV, slots),
                bt=torch.randperm(N * 4, generator=torch.Generator().manual_seed(1)).view(N, 4).int().to(gpu),
                lens=torch.tensor([1, 64, 17, 33, 50], dtype=torch.int32, device=gpu), D=D)


def _decode(i, **kw):
    return paged_spike_attn_decode(i["q"], i["k"], i["v"], i["bt"], i["lens"], i["D"], BS, HQ, HKV, **kw)


def test_module_is_built_and_bound():
    assert _lib.native() is not None


@pytest.mark.parametrize("D", [64, 128, 40])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_same_outputs(gpu, D, dtype):
    i = _inputs(gpu, D)
    native = _lib.native()
    out = torch.empty((T, N, HQ, D), dtype=dtype, device=gpu)
    assert native.decode_attn(i["q"], i["k"], i["v"], i["bt"], i["lens"], D, BS, HQ, HKV, out, dtype, None) is out
    got = _decode(i, dtype=dtype)
    # long tables: a workspace for split contexts
    wide = dict(i, bt=i["bt"].repeat(1, 600))
    split = _decode(wide, dtype=dtype)
    assert got.dtype == dtype and got.shape == out.shape
    with _without_native():
        assert torch.equal(got, _decode(i, dtype=dtype)) and torch.equal(out, got)
        assert torch.equal(split, _decode(wide, dtype=dtype))

    x = torch.randn((T, 7, 3, D), device=gpu).to(dtype)
    b, th = torch.full((D,), 0.9, device=gpu), torch.full((D,), 1.0, device=gpu)
    packed = torch.zeros((T, 7, 3, -(-D // 32)), dtype=torch.int32, device=gpu)
    cache = torch.zeros((T, 3, 40, -(-D // 32)), dtype=torch.int32, device=gpu)
    slots = torch.arange(7, device=gpu) * 5
    sites = [(x, b, th, packed, False), (x, b, th, cache, True)]
    assert native.lif_sites(sites, slots) is True
    s, u = lif_multistep(x, b, th, return_membrane=True)
    assert native.lif(x, b, th, False) is not None
    with _without_native():
        p2, c2 = torch.zeros_like(packed), torch.zeros_like(cache)
        lif_pack_write_sites([(x, b, th, p2, False), (x, b, th, c2, True)], slots)
        s2, u2 = lif_multistep(x, b, th, return_membrane=True)
    assert torch.equal(packed, p2) and torch.equal(cache, c2) and torch.equal(s, s2) and torch.equal(u, u2)
    assert u.shape == x.shape[1:] and s.shape == x.shape

    o = [torch.zeros((T, N + 2, HQ, D), dtype=dtype, device=gpu) for _ in range(2)]
    chunks = [(0, 2, 2, 30, i["bt"][1]), (2, 4, 3, 0, None)]
    assert native.prefill(i["q"], i["k"], i["v"], chunks, o[0], D, BS) is True
    with _without_native():
        paged_spike_attn_prefill(i["q"], i["k"], i["v"], chunks, o[1], D, BS)
    assert torch.equal(*o)


def test_other_forms_end_as_without_it(gpu):
    i = _inputs(gpu)
    native = _lib.native()
    want = _decode(i)
    args = lambda **c: {**i, **c}
    for same in (args(bt=i["bt"].long()), args(lens=i["lens"].long()), args(bt=i["bt"].repeat(1, 2)[:, :4]),
                 args(lens=i["lens"].repeat_interleave(2)[::2])):
        assert torch.equal(_decode(same), want)
    q2 = torch.zeros((T, N, 2 * HQ, 2), dtype=torch.int32, device=gpu)[:, :, ::2]
    q2.copy_(i["q"])
    assert torch.equal(_decode(args(q=q2)), want)  # a strided view, taken as it is
    empty = _decode(dict(i, q=i["q"][:, :0], bt=i["bt"][:0], lens=i["lens"][:0]))
    assert empty.shape == (T, 0, HQ, 64)
    bad = [args(q=i["q"].cpu()), args(q=i["q"].long()), args(k=i["k"][:2], v=i["v"][:2]), args(k=i["k"][:, :, :-1]),
           args(lens=i["lens"][:2]), args(q=i["q"][..., :1])]
    for b in bad:
        assert native.decode_attn(b["q"], b["k"], b["v"], b["bt"], b["lens"], 64, BS, HQ, HKV, None, torch.float32,
                                  None) is None
        with pytest.raises(ValueError):
            _decode(b)
    with pytest.raises(ValueError):
        _decode(i, out=torch.empty((T, N, HQ, 32), device=gpu))
    wide = dict(i, bt=i["bt"].repeat(1, 600))
    with pytest.raises(ValueError):
        _decode(wide, workspace=torch.empty(8, dtype=torch.uint8, device=gpu))
    x = torch.randn((T, 6, 64), device=gpu)
    b, th = torch.full((64,), 0.9, device=gpu), torch.full((64,), 1.0, device=gpu)
    ref = lif_multistep(x, b, th)
    assert torch.equal(lif_multistep(x, b.double(), th.view(1, 64)), ref)
    assert torch.equal(lif_multistep(x.transpose(1, 2).contiguous().transpose(1, 2), b, th), ref)
    assert torch.equal(lif_multistep(x, b.bfloat16().float(), th.bfloat16()),
                       lif_multistep(x, b.bfloat16(), th.bfloat16()))
    with pytest.raises(AssertionError):
        lif_multistep(x, b[:32], th)
    with pytest.raises(ValueError):
        lif_multistep(x.double(), b, th)
    with pytest.raises(ValueError):
        lif_pack_write_sites([], None)


@pytest.mark.parametrize("n", [3, 70])
def test_decoder_operators(gpu, n):
    """A decoder layer over a prompt: the same words and hidden states with and
    without the module, and each operator takes the model's arguments."""
    from spikeinfer_amd.attention import AttentionMetadata
    from spikeinfer_amd.kernels import decoder_ops as ops
    from spikeinfer_amd.model import SpikingDecoder, SpikingQwenConfig
    from spikeinfer_amd.spike_cache import PagedSpikeCache

    cfg = SpikingQwenConfig(vocab_size=512, num_hidden_layers=1)
    model = SpikingDecoder(cfg, device=gpu, seed=3)
    ids, pos = torch.arange(n, device=gpu), torch.arange(n, device=gpu)
    meta = AttentionMetadata(slot_mapping=pos + 5, block_size=16, prefill_query_starts=[0], prefill_query_lens=[n],
                             prefill_context_lens=[0], prefill_block_tables=[torch.arange(6, device=gpu).int()])
    taken, names = set(), ("embed_rmsnorm", "add_rmsnorm", "rmsnorm_mean_t", "lif_gate_mul", "linear_decode",
                           "mlp_gate_lif", "qkv_rope_lif_pack", "prefill")
    real = _lib.native()

    class Spy:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(real, name)(*a)
                if r is not None:
                    taken.add(name)
                return r
            return call

    outs = []
    for module in (Spy(), None):
        _lib._native = module
        try:
            cache = PagedSpikeCache(1, 4, 2, 64, 8, 16, device=gpu)
            hidden = model.forward_paged(ids, pos, cache.layers, meta)
            outs.append((hidden, model.compute_logits(hidden[-1:]), cache.k[0], cache.v[0]))
            if n > 64:
                x = torch.ones((4, 8, 896), device=gpu, dtype=torch.bfloat16)
                ops.mlp_gate_lif(x, model.layers[0].w_gu_packed, model.layers[0].lif_gate_beta,
                                 model.layers[0].lif_gate_th)
            else:
                ops.lif_gate_mul(torch.ones((4, n, 2 * 4864), device=gpu, dtype=torch.bfloat16),
                                 model.layers[0].lif_gate_beta, model.layers[0].lif_gate_th)
        finally:
            _lib._native = real
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    assert taken == set(names)


def test_on_another_stream_and_in_a_graph(gpu):
    """The launch goes to the stream that is current when it is made."""
    i = _inputs(gpu)
    want = _decode(i)
    out = torch.zeros_like(want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _decode(i, out=out)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _decode(i, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
