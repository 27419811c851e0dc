"""GPU: a user turn of a few hundred tokens after a long context, whose prefill splits every
item's key range over a full round of workgroups, against the oracle; the allocation-free entry
point makes the same split (bit-identical); a capture without a reserved workspace scans whole
key ranges instead. Tolerances as for every f16 / q8 attention (relative 2e-3)."""
import gc

import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from bitgpu_amd._lib import GpuOutOfMemoryError, check, lib
from oracle import ref
from tests.gpu_helpers import cached_values, run_attention, run_attention_noalloc, t
from tests.test_gpu_sink_copy import _ring
from tests.test_gpu_split_prefill import _case, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,H,KV,D,ctx,S,gate", [
    ("q8", 32, 8, 128, 6001, 333, False),    # 88 items in five parts of 20 steps, the last shorter
    ("f16", 16, 8, 128, 5000, 97, False),    # 16 items in many parts
    ("q8", 24, 4, 256, 3001, 300, True),     # 60 items in four parts, gated
    ("f16", 32, 8, 128, 2999, 250, False),   # 64 items
])
def test_turn_after_context(dev, dtype, H, KV, D, ctx, S, gate):
    c, _, q, g = _case(dtype, H, KV, D, ctx + S, S, seed=ctx + S, gate=gate)
    scale = 1.0 / np.sqrt(D)
    out = run_attention(c, 0, q, ctx, scale=scale, gate=g)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    _check(out, ref.gated_attention(q, kk, vv, g, ctx) if gate else ref.attention(q, kk, vv, ctx, scale=scale))
    assert np.array_equal(run_attention_noalloc(c, 0, q, ctx, scale=scale, gate=g), out)
    c.close()


def test_turn_captured_without_reserve(dev):
    H, KV, D, ctx, S = 32, 8, 128, 5000, 200
    c, _, q, _ = _case("f16", H, KV, D, ctx + S, S, seed=3, gate=False)
    qt, out = t(q), torch.empty(S, H, D, device="cuda")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        E.attention(c, 0, qt, S, H, ctx, out=out)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    want = ref.attention(q, kk, vv, ctx)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _check(out.cpu().numpy(), want)
    c.close()


def test_split_partials_stay_within_their_bound(dev):
    """Plans of growing partials use one buffer of 33 MiB, as the header states (the memory in use
    grows by no more, rounded up to the allocator's pages)."""
    H, KV, D, ctx = 32, 8, 128, 16000
    q, out = torch.randn(333, H, D, device="cuda"), torch.empty(333, H, D, device="cuda")
    for _ in range(2):  # the first cache also loads the kernels
        c = E.KvCache(1, KV, D, "f16", max_seq_len=ctx + 64, capacity=ctx + 64)
        gc.collect()  # no other cache is given back between the two readings
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for S, at in ((100, 1000), (64, ctx), (333, 12001)):   # 8, 16 and 27.5 MiB of partials
            E.attention(c, 0, q[:S], S, H, at, out=out[:S])
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]
        c.close()
    assert 33 << 20 <= used <= 35 << 20, used


def test_reserve_without_memory(dev, monkeypatch):
    """Where an f32 or sink-mode launch can do without the partials and the copy, a reserve that
    cannot have them is no error; f16 and q8 report it, and the plain q8 prefill, which needs its
    copy, too."""
    H, KV, D, ctx, S = 32, 8, 128, 2000, 150

    def reserve(c, S):
        check(lib().bg_attention_reserve(c.handle, S, H))
    monkeypatch.setenv("BG_FAULT_PREFILL_ALLOC", "1")
    c, _, q, _ = _case("f32", H, KV, D, ctx + S, S, seed=6, gate=False)
    reserve(c, S)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    want = ref.attention(q, kk, vv, ctx)
    assert np.abs(run_attention(c, 0, q, ctx) - want).max() <= 1e-4
    c.close()
    c, q, want = _ring("f16", H, KV, D, 1000, (300,), 700, 100, "slot")
    # (the copy is let go; the partials of an f16 cache are reported as before)
    with pytest.raises(GpuOutOfMemoryError, match="split prefill"):
        reserve(c, 100)
    _check(run_attention(c, 0, q, 700), want)
    c.close()
    c, _, q, _ = _case("q8", H, KV, D, 700, 60, seed=7, gate=False)
    with pytest.raises(GpuOutOfMemoryError, match="split prefill"):
        reserve(c, 60)
    with pytest.raises(GpuOutOfMemoryError, match="f16 copy"):
        reserve(c, 128)
    kk, vv = cached_values(c, 0, 0, 700)
    _check(run_attention(c, 0, q, 640), ref.attention(q, kk, vv, 640))
    with pytest.raises(GpuOutOfMemoryError):
        run_attention(c, 0, np.repeat(q, 3, 0), 500)
    monkeypatch.delenv("BG_FAULT_PREFILL_ALLOC")
    reserve(c, 128)
    c.close()
