"""GPU: f32 prefill at head_dim 128 over its plans -- waves sharing 32, 64 and 128 rows, key ranges
split over workgroups, heads per kv head that do not divide 32, wrapped sink rings -- against the
oracle (max-abs 1e-4, the bar for f32 storage)."""
import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from oracle import ref
from tests.gpu_helpers import cached_values, run_attention, run_attention_noalloc, t
from tests.test_gpu_sink_copy import _ring
from tests.test_gpu_split_prefill import _case
from tests.test_host import f32_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,ctx,S,gate", [
    (16, 8, 0, 9, False),       # 18 rows a kv head over one step: 128-row items, keys through LDS
    (16, 8, 24, 9, True),       # one more key than a step: a partial 32-row item
    (12, 4, 0, 32, True),       # 96 rows over one step: the most that kernel takes
    (16, 4, 7, 25, False),      # 100 rows over one step: 32-row items
    (16, 8, 0, 333, True),      # 32-row items, a ragged end
    (24, 8, 0, 129, False),     # 3 heads a kv head: queries across row groups
    (12, 1, 700, 40, False),    # 12 heads a kv head
    (100, 1, 50, 3, True),      # 100 heads: a query an item
    (32, 8, 5000, 9, False),    # a verify after a long context: parts over workgroups
    (16, 2, 4001, 70, True),
    (32, 8, 2000, 150, False),
])
def test_f32_plans(dev, H, KV, ctx, S, gate):
    c, _, q, g = _case("f32", H, KV, 128, ctx + S, S, seed=H + ctx + S, gate=gate)
    out = run_attention(c, 0, q, ctx, gate=g)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    want = ref.gated_attention(q, kk, vv, g, ctx) if gate else ref.attention(q, kk, vv, ctx)
    assert np.abs(out - want).max() <= 1e-4
    assert np.array_equal(run_attention_noalloc(c, 0, q, ctx, gate=g), out)
    c.close()


def test_f32_wide_rows(dev):
    """128-row items, a wave its own rows (a long prompt), on a sample of the rows."""
    H, KV, S = 32, 8, 2048
    c, _, q, _ = _case("f32", H, KV, 128, S, S, seed=1, gate=False)
    out = run_attention(c, 0, q, 0)
    kk, vv = cached_values(c, 0, 0, S)
    for r in (0, 31, 777, 2040):
        want = ref.attention(q[r:r + 8], kk[:r + 8], vv[:r + 8], r)
        assert np.abs(out[r:r + 8] - want).max() <= 1e-4
    c.close()


@pytest.mark.parametrize("window,moves,fill,S,mode", [
    (1000, (300,), 700, 60, "slot"), (1000, (900,), 700, 100, "absolute"), (1020, (316,), 960, 64, "slot")])
def test_f32_sink_ring(dev, window, moves, fill, S, mode):
    c, q, want = _ring("f32", 32, 8, 128, window, moves, fill, S, mode)
    assert np.abs(run_attention(c, 0, q, fill) - want).max() <= 1e-4
    c.close()


@pytest.mark.parametrize("H,KV,D,fill,S,mode", [
    (32, 8, 128, 0, 333, "slot"), (16, 4, 128, 650, 70, "absolute"), (8, 2, 256, 0, 150, "slot")])
def test_f32_sink_prompt_before_any_eviction(dev, H, KV, D, fill, S, mode):
    """The ring's origin has not moved: the causal bound, as for the plain cache."""
    c, q, want = _ring("f32", H, KV, D, 1000, (), fill, S, mode)
    out = run_attention(c, 0, q, fill)
    assert np.abs(out - want).max() <= 1e-4
    assert np.array_equal(run_attention_noalloc(c, 0, q, fill), out)
    c.close()


def _plan(KV, S, H, pos_base, **ring):
    """(waves sharing 32 rows, parts) and queries an item of the launch on this GPU."""
    rc, (ks, QB, parts, _) = f32_plan(KV, S, H, pos_base, cus=torch.cuda.get_device_properties(0).multi_processor_count, **ring)
    assert rc == 0
    return (ks, parts), QB


@pytest.mark.parametrize("H,KV,ctx,S,gate,ks,parts", [
    (32, 8, 1000, 90, True, 1, 9),     # four row groups an item; the last item's groups end before its last part
    (16, 4, 9000, 200, False, 1, 9),
    (32, 8, 16000, 600, False, 1, 3),
    (24, 8, 1500, 120, False, 1, 9),   # 3 heads a kv head: a query's rows in two groups
    (24, 8, 800, 121, True, 2, 5),
    (16, 2, 1000, 104, False, 2, 9),   # two row groups an item
])
def test_f32_row_groups_in_parts(dev, H, KV, ctx, S, gate, ks, parts):
    """Waves of one or two row groups whose keys are split over workgroups, on a sample of the rows
    (ends and row group borders among them)."""
    plan, QB = _plan(KV, S, H, ctx)
    assert plan == (ks, parts)
    c, _, q, g = _case("f32", H, KV, 128, ctx + S, S, seed=ctx + S, gate=gate)
    out = run_attention(c, 0, q, ctx, gate=g)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    for r in sorted({0, 7, 8, 10, 11, QB - 1, QB, S // 2, S - 9, S - 2, S - 1}):
        a = (q[r:r + 1], kk[:ctx + r + 1], vv[:ctx + r + 1])
        want = ref.gated_attention(*a, g[r:r + 1], ctx + r) if gate else ref.attention(*a, ctx + r)
        assert np.abs(out[r:r + 1] - want).max() <= 1e-4, r
    assert np.isfinite(out).all() and np.array_equal(run_attention_noalloc(c, 0, q, ctx, gate=g), out)
    c.close()


@pytest.mark.parametrize("H,KV,window,moves,fill,S,mode,ks,parts", [
    (32, 8, 1000, (300,), 225, 769, "slot", 1, 1),
    (32, 8, 1000, (300,), 502, 321, "absolute", 2, 1),
    (24, 4, 2000, (700,), 1911, 83, "slot", 1, 16),
    (32, 8, 4096, (1500,), 4063, 27, "absolute", 2, 13),
])
def test_f32_ring_row_groups(dev, H, KV, window, moves, fill, S, mode, ks, parts):
    c, q, want = _ring("f32", H, KV, 128, window, moves, fill, S, mode)
    assert _plan(KV, S, H, fill, window=window + 4, sinks=4, head=c.ring_state()[0])[0] == (ks, parts)
    out = run_attention(c, 0, q, fill)
    assert np.abs(out - want).max() <= 1e-4
    assert np.array_equal(run_attention_noalloc(c, 0, q, fill), out)
    c.close()


def test_f32_captured_without_reserve(dev):
    """No buffer for partials can be had under capture: one part, on the rows planned for that."""
    H, KV, ctx, S = 16, 4, 9000, 200
    c, _, q, _ = _case("f32", H, KV, 128, ctx + S, S, seed=4, gate=False)
    qt, out = t(q), torch.empty(S, H, 128, device="cuda")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        E.attention(c, 0, qt, S, H, ctx, out=out)
    kk, vv = cached_values(c, 0, 0, ctx + S)
    rows = [0, 7, 8, 31, 32, 100, 199]
    want = np.concatenate([ref.attention(q[r:r + 1], kk[:ctx + r + 1], vv[:ctx + r + 1], ctx + r) for r in rows])
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.isfinite(got).all() and np.abs(got[rows] - want).max() <= 1e-4
    c.close()
