"""Appends of many 16-bit rows, whose whole pages are stored through LDS, against the oracle
byte for byte: chunks that start on and off page boundaries, with runs broken at every place
(skipped and out-of-range slots, swapped and scattered rows, gaps), strided sources, and row
counts on both sides of the kernel choice."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import paged_kv as orc

pytestmark = pytest.mark.gpu


def _slots(n, seed, kind):
    """Slots of n tokens: chunks on consecutive pages of a permutation, then broken."""
    r = np.random.default_rng(seed)
    pages = r.permutation(n // 8 + 64)
    out, at = [], 0
    while len(out) < n:
        start, size = (0, 512) if kind == "aligned" else (int(r.integers(0, 16)), int(r.integers(1, 200)))
        pos = start + np.arange(min(size, n - len(out)))
        out += list(pages[at + pos // 16] * 16 + pos % 16)
        at += int(pos[-1]) // 16 + 1
        assert at < len(pages) - 1
    s = np.array(out, dtype=np.int32)
    if kind == "broken":
        pick = r.permutation(n)
        s[pick[:n // 50]] = -1
        s[pick[n // 50:n // 40]] = len(pages) * 16 + 5  # past the pool
        a, b = pick[-n // 20:-n // 40], pick[-n // 40:]
        m = min(len(a), len(b))
        s[a[:m]], s[b[:m]] = s[b[:m]].copy(), s[a[:m]].copy()
    elif kind == "scattered":
        s = s[r.permutation(n)]
    return torch.from_numpy(s), len(pages)


@pytest.mark.parametrize("kind", ["aligned", "ragged", "broken", "scattered"])
@pytest.mark.parametrize("n,hkv,d", [(2047, 8, 128), (2048, 8, 128), (2061, 9, 128), (4100, 8, 64), (2500, 13, 128),
                                     (8192, 4, 256), (8205, 5, 256), (16500, 1, 128)])
def test_many_rows_bit_exact(iva, dev, kind, n, hkv, d):
    slots, n_pages = _slots(n, n + hkv, kind)
    gen = torch.Generator().manual_seed(n)
    rows = torch.randint(-32768, 32768, (n, 2, hkv, d), dtype=torch.int16, generator=gen)
    src = rows.to(dev).view(torch.float16)  # k and v rows interleaved: strided sources
    ks, vs = iva.pool_shapes(n_pages, hkv, d, 16, torch.float16)
    k_pool = torch.full(ks, 0x1234, dtype=torch.int16, device=dev).view(torch.float16)
    v_pool = torch.full(vs, 0x1234, dtype=torch.int16, device=dev).view(torch.float16)
    iva.kv_append(src[:, 0], src[:, 1], k_pool, v_pool, slots.to(dev))
    ok, ov = orc.empty_pools(n_pages, hkv, d, 16, np.uint16, fill=0x1234)
    orc.append(ok, ov, rows[:, 0].contiguous().numpy().view(np.uint16),
               rows[:, 1].contiguous().numpy().view(np.uint16), slots.numpy())
    assert np.array_equal(k_pool.view(torch.int16).cpu().numpy().view(np.uint16), ok)
    assert np.array_equal(v_pool.view(torch.int16).cpu().numpy().view(np.uint16), ov)
