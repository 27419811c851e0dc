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
    ("f32", 24, 8, 128, 128, 2049, False),  # past f32's line (65,536 rows)
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
