"""GPU: whole-snapshot save and restore (bg_kv_save / bg_kv_load) byte for byte against the
per-region export: pieces that fill a staging slot and remainders, a base, rings whose origin has
moved, head_dim 256, several threads at once; argument errors."""
import threading

import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from bitgpu_amd._lib import BG_E_INVALID, BitgpuError, check, lib

pytestmark = pytest.mark.gpu


def _filled(dtype, layers, KV, D, n, roll=False, seed=0):
    kw = dict(overflow="sinks", sink_tokens=4) if roll else {}
    c = E.KvCache(layers, KV, D, dtype, max_seq_len=n + 40, capacity=n + 40, **kw)
    if roll:
        c.evict(n + 40, n // 3)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for li in range(layers):
        for w in (0, 1):
            c.append_kv(torch.randn(n, KV, D, generator=g, device="cuda"), w, li, n * KV, 0)
    return c


def _by_region(c, n, base=0):
    return b"".join(c.export_rows(li, r, base, n - base) for li in range(c.n_layers) for r in c._regions())


@pytest.mark.parametrize("dtype,layers,KV,D,n,base,roll", [
    ("q8", 2, 8, 128, 2500, 0, False),    # three slots a layer, the last one short
    ("q8", 3, 8, 128, 333, 17, False),
    ("f16", 2, 8, 128, 1100, 0, True),
    ("q8", 2, 4, 256, 777, 0, True),
    ("f32", 11, 8, 128, 300, 1, False),   # more pieces than slots
    ("f32", 1, 1, 256, 1, 0, False),
])
def test_save_and_restore_whole(dev, dtype, layers, KV, D, n, base, roll):
    a = _filled(dtype, layers, KV, D, n, roll)
    data = a.save_snapshot(n, base)
    assert data == _by_region(a, n, base)
    b = _filled(dtype, layers, KV, D, n, roll, seed=1)
    before = _by_region(b, n)
    b.restore_snapshot(data if n % 2 else bytearray(data), n, base)
    assert b.save_snapshot(n, base) == data
    if base:
        assert b.save_snapshot(base) == _by_region(b, base) and _by_region(b, n) != before
    a.close()
    b.close()


def test_save_from_threads(dev):
    caches = [_filled("q8", 4, 8, 128, 900, seed=s) for s in range(3)]
    torch.cuda.synchronize()
    want, got = [_by_region(c, 900) for c in caches], [None] * 3

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = caches[i].save_snapshot(900)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert got == want
    [c.close() for c in caches]


def test_save_arguments(dev):
    c = _filled("q8", 1, 8, 128, 64)
    buf = np.zeros(64 * 2304, np.uint8)
    for args in ((0, 64, buf.ctypes.data, buf.nbytes - 1), (0, 64, None, buf.nbytes), (60, 64, buf.ctypes.data, buf.nbytes),
                 (-1, 64, buf.ctypes.data, buf.nbytes), (0, -1, buf.ctypes.data, 0)):
        for fn in (lib().bg_kv_save, lib().bg_kv_load):
            with pytest.raises(BitgpuError) as e:
                check(fn(c.handle, *args, None))
            assert e.value.code == BG_E_INVALID
    assert c.save_snapshot(0) == b""
    c.restore_snapshot(b"", 0)
    c.close()


def test_restore_of_nothing_past_the_cache_is_refused(dev):
    c = _filled("q8", 1, 8, 128, 64)
    c.restore_snapshot(b"", 104, 104)  # the end of the cache
    with pytest.raises(BitgpuError) as e:
        c.restore_snapshot(b"", 105, 105)
    assert e.value.code == BG_E_INVALID
    c.close()


def test_positions_wider_than_a_staging_slot(dev):
    """2,100 kv heads of f32: 2.15 MB a position, past a 2 MiB slot; goes region by region."""
    a = _filled("f32", 1, 2100, 128, 3)
    data = a.save_snapshot(3)
    assert data == _by_region(a, 3)
    b = _filled("f32", 1, 2100, 128, 3, seed=1)
    b.restore_snapshot(data, 3)
    assert _by_region(b, 3) == data
    a.close()
    b.close()
