"""GPU: the prologue's row layouts (one, two and four row loads a wave) give the same bits for a
row: positions written one step at a time (one load a wave) equal the same positions written as
one batch that the other layouts take, q_out and every stored byte, at batch ends that leave a
partial wave, with and without Q, K rotation and a partial rotary width."""
import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from tests.gpu_helpers import rope_dev, t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,H,KV,D,rot,S,roll", [
    ("f16", 32, 8, 128, 128, 207, False),   # just past the one-load line (8,192 rows)
    ("q8", 12, 3, 128, 96, 549, False),     # rows that share no position a wave; a width through LDS
    ("q8", 24, 4, 256, 64, 293, False),
    ("f16", 32, 8, 128, 128, 211, True),
    ("f32", 24, 8, 128, 128, 2049, False),  # past f32's line (1.8 M values of V)
    ("f32", 12, 3, 256, 64, 2341, False),
])
def test_layouts_give_the_same_bits(dev, dtype, H, KV, D, rot, S, roll):
    rng = np.random.default_rng(S)
    kw = dict(overflow="sinks", sink_tokens=4) if roll else {}
    caches = [E.KvCache(1, KV, D, dtype, max_seq_len=S + 70, capacity=S + 70, **kw) for _ in range(2)]
    cos, sin, _, _ = rope_dev(1e6, rot, S + 70)
    q, k, v = (t(rng.standard_normal((S, h, D)).astype(np.float32)) for h in (H, KV, KV))
    gq, gk = (t((1 + 0.1 * rng.standard_normal(D)).astype(np.float32)) for _ in range(2))
    p = 3
    whole = E.qkv_prologue(caches[0], 0, q, k, v, S, H, gq, gk, 1e-6, cos, sin, rot, p, p)
    step = max(1, min(S, 5000 // (H + KV)))
    parts = [E.qkv_prologue(caches[1], 0, q[i:i + step], k[i:i + step], v[i:i + step], len(q[i:i + step]), H, gq, gk, 1e-6,
                            cos, sin, rot, p + i, p + i) for i in range(0, S, step)]
    torch.cuda.synchronize()
    assert torch.equal(whole.view(torch.int32), torch.cat(parts).view(torch.int32))
    assert caches[0].save_snapshot(S + p) == caches[1].save_snapshot(S + p)
    [c.close() for c in caches]


@pytest.mark.parametrize("dtype,H,D,S", [("f16", 32, 128, 300), ("q8", 24, 256, 2800), ("f32", 32, 128, 2100)])
def test_queries_alone(dev, dtype, H, D, S):
    """Q without K and V, on few and many rows of every storage type: the bits of the whole call, and
    nothing written to the cache."""
    c = E.KvCache(1, 4, D, dtype, max_seq_len=S, capacity=S)
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(S, h, D, generator=g, device="cuda") for h in (H, 4, 4))
    gamma = torch.rand(D, generator=g, device="cuda") + 0.5
    cos, sin, _, _ = rope_dev(1e6, D, S)
    before = c.save_snapshot(S)
    alone = E.qkv_prologue(c, 0, q, None, None, S, H, gamma, None, 1e-6, cos, sin, D, 0, 0)
    assert c.save_snapshot(S) == before
    whole = E.qkv_prologue(c, 0, q, k, v, S, H, gamma, gamma, 1e-6, cos, sin, D, 0, 0)
    assert torch.equal(alone.view(torch.int32), whole.view(torch.int32))
    c.close()
