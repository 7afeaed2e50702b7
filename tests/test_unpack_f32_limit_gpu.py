"""fp32 outputs of a table with more tiles than the allocation-free entry point's scratch holds one to
a workgroup: two are taken then, and the bytes are the same. A widen of 8.5 G elements and, beside it, short
dequants of an odd number of tiles (4096 elements), whose last workgroup's second tile lies past the
region: rows wider than 2 KiB of output, narrower ones, and rows shorter than a chunk."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import squareq as oq
from stagehand_amd.unpack import KIND_BF16_F32, KIND_I8_ROWSCALE_F32, make_descs, unpack_noalloc

pytestmark = pytest.mark.gpu


def test_two_tiles_to_a_workgroup():
    n = 4096 * 2064384 + 4097
    shapes = [(31, 1155), (91, 101), (4000, 3)]
    rng = np.random.default_rng(3)
    q = [rng.integers(-127, 128, shape, dtype=np.int8) for shape in shapes]
    s = [np.exp(rng.normal(-6, 0.5, rows)).astype(np.float32) for rows, _ in shapes]
    n_q = sum(x.size for x in q)
    src = torch.empty(2 * n + n_q, dtype=torch.uint8, device="cuda")
    wide = src[:2 * n].view(torch.bfloat16)
    step = 1 << 30
    for at in range(0, n, step):
        m = min(step, n - at)
        wide[at:at + m].copy_(torch.arange(at, at + m, device="cuda", dtype=torch.int64).remainder_(65521).float())
    descs = [(KIND_BF16_F32, 0, 0, n // 4097, 4097, 0, 0),
             (KIND_BF16_F32, 2 * (n // 4097) * 4097, 4 * (n // 4097) * 4097, 1, n % 4097, 0, 0)]
    at, row, spans = 0, 0, []
    for (rows, cols), x in zip(shapes, q):
        assert -(-x.size // 4096) % 2 == 1
        src[2 * n + at:2 * n + at + x.size].copy_(torch.from_numpy(x.view(np.uint8).reshape(-1)).cuda())
        descs.append((KIND_I8_ROWSCALE_F32, 2 * n + at, 4 * (n + at), rows, cols, 0, row))
        spans.append((n + at, n + at + x.size))
        at, row = at + x.size, row + rows
    dst = torch.full((n + n_q + 64,), -7.0, device="cuda")
    unpack_noalloc(make_descs(descs), src, dst, torch.from_numpy(np.concatenate(s)).cuda())
    for at in range(0, n, step):
        m = min(step, n - at)
        assert torch.equal(dst[at:at + m], wide[at:at + m].float()), at
    for (rows, cols), x, scale, (a, b) in zip(shapes, q, s, spans):
        np.testing.assert_array_equal(dst[a:b].cpu().numpy().reshape(rows, cols).view(np.uint32),
                                      oq.dequant_rows(x, scale, None, rows, cols, out="float32").view(np.uint32))
    assert bool((dst[n + n_q:] == -7.0).all())
