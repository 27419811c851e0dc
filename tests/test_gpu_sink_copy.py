"""GPU: sink-mode prefill on the f16 copy of rotated keys. The copy's rotation and the staging's
(the allocation-free entry point, and a capture without a reserved copy) share their arithmetic,
so the outputs are equal bit for bit; both are checked against the oracle over the stored values
(relative 2e-3). Ring origins and fills put the room eviction left in one piece or across the
ring's end, the seam inside a step, on its first slot, right behind the sinks."""
import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from oracle import ref
from tests.gpu_helpers import cached_values, fill_cache_raw, rope_dev, run_attention, run_attention_noalloc, t
from tests.test_gpu_split_prefill import _check

pytestmark = pytest.mark.gpu


def _ring(dtype, H, KV, D, window, moves, fill, S, mode="slot", seed=0):
    rng = np.random.default_rng(seed + fill + S)
    m = 4 + window
    c = E.KvCache(1, KV, D, dtype, max_seq_len=m, overflow="sinks", sink_tokens=4, rope_positions=mode)
    for need in moves:
        c.evict(m, need)
    evicted = c.ring_state()[1]
    cos_d, sin_d, cos, sin = rope_dev(1e6, D, m + (evicted if mode == "absolute" else 0))
    c.set_rope(cos_d, sin_d)
    k, v = (rng.standard_normal((fill + S, KV, D)).astype(np.float32) for _ in range(2))
    fill_cache_raw(c, 0, k, v)
    q = rng.standard_normal((S, H, D)).astype(np.float32)
    kk, vv = cached_values(c, 0, 0, fill + S)
    at = np.arange(fill + S)
    at[4:] += evicted if mode == "absolute" else 0
    h = D // 2
    cs, sn = cos[at][:, None], sin[at][:, None]
    kr = np.concatenate([kk[..., :h] * cs - kk[..., h:] * sn, kk[..., h:] * cs + kk[..., :h] * sn], -1)
    return c, q, ref.attention(q, kr.astype(np.float32), vv, fill)


@pytest.mark.parametrize("dtype,D,window,moves,fill,S,mode", [
    ("f16", 128, 1000, (), 600, 90, "slot"),            # before any eviction
    ("f16", 128, 1000, (300,), 700, 100, "slot"),       # room of three whole steps behind the seam
    ("q8", 128, 1000, (900,), 700, 100, "slot"),        # room across the ring's end
    ("f16", 128, 1020, (316,), 1024 - 64, 64, "slot"),  # full, seam on a step's first slot
    ("q8", 128, 997, (997, 251), 500, 333, "absolute"),
    ("f16", 128, 997, (996,), 300, 70, "absolute"),     # seam on the last slot
    ("f16", 256, 640, (200,), 450, 120, "slot"),
    ("q8", 256, 640, (639,), 300, 77, "slot"),
])
def test_sink_prefill_copy_equals_staging(dev, dtype, D, window, moves, fill, S, mode):
    H, KV = (32, 8) if D == 128 else (12, 2)
    c, q, want = _ring(dtype, H, KV, D, window, moves, fill, S, mode)
    out = run_attention(c, 0, q, fill)
    _check(out, want)
    assert np.array_equal(run_attention_noalloc(c, 0, q, fill), out)
    c.close()


@pytest.mark.parametrize("dtype,H,KV,D,window,moves,fill,S", [
    ("f16", 32, 8, 128, 700, (200,), 350, 17),     # nine steps, room left out: three parts of three
    ("q8", 32, 8, 128, 700, (), 660, 16),          # six parts of two steps, the last of one
    ("f16", 16, 1, 128, 1500, (400,), 1400, 7),    # twelve parts: the merge of a workgroup a slot
    ("q8", 24, 4, 256, 700, (600,), 350, 9),
    ("f16", 64, 8, 128, 4096, (1500,), 4050, 16),  # 128 rows, parts of three
])
def test_one_block_in_parts_of_rotating_steps(dev, dtype, H, KV, D, window, moves, fill, S):
    """One query block of more rows than the decode kernel takes: no copy, every step rotates its keys,
    parts down to two steps."""
    c, q, want = _ring(dtype, H, KV, D, window, moves, fill, S)
    out = run_attention(c, 0, q, fill)
    _check(out, want)
    assert np.array_equal(run_attention_noalloc(c, 0, q, fill), out)
    c.close()


def test_sink_prefill_captured_without_reserve(dev):
    H, KV, D, fill, S = 32, 8, 128, 1500, 160
    c, q, want = _ring("f16", H, KV, D, 2000, (700,), fill, S)
    qt, out = t(q), torch.empty(S, H, D, device="cuda")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        E.attention(c, 0, qt, S, H, fill, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _check(out.cpu().numpy(), want)
    c.close()


@pytest.mark.parametrize("dtype,kw", [("f16", dict(overflow="sinks", sink_tokens=4)), ("q8", {})])
def test_first_copy_does_not_wait_for_other_streams(dev, dtype, kw):
    """The first prefill of a cache allocates its copy and returns while another stream is busy
    (with 40 products of 8192 x 8192 f32 matrices, a few hundred ms), and is right."""
    H, KV, D, S = 32, 8, 128, 200
    cos, sin, _, _ = rope_dev(1e6, D, 1024)
    q = torch.randn(S, H, D, device="cuda")
    k, v = (torch.randn(S, KV, D, device="cuda") for _ in range(2))
    m = torch.randn(8192, 8192, device="cuda")
    p = m @ m
    outs = []
    for busy in (False, True):  # the first pass also loads the kernels
        c = E.KvCache(1, KV, D, dtype, max_seq_len=1024, capacity=1024, **kw)
        if kw:
            c.set_rope(cos, sin)
        c.append_kv(k, 0, 0, S * KV, 0)
        c.append_kv(v, 1, 0, S * KV, 0)
        out = torch.empty_like(q)
        torch.cuda.synchronize()
        other, done = torch.cuda.Stream(), torch.cuda.Event()
        if busy:
            with torch.cuda.stream(other):
                for _ in range(40):
                    torch.matmul(m, m, out=p)
                done.record()
        E.attention(c, 0, q, S, H, 0, out=out)
        waited = done.query()
        torch.cuda.synchronize()
        assert not (busy and waited)
        outs.append(out.clone())
        c.close()
    assert torch.equal(*outs)
