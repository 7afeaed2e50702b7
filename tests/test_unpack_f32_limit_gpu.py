"""fp32 outputs of a table with more tiles than the allocation-free entry point's scratch holds one to
a workgroup: two are taken then, and the bytes are the same (a widen of 8.5 G elements and, beside it,
a short dequant of odd rows, whose last workgroup has one tile)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import squareq as oq
from stagehand_amd.unpack import KIND_BF16_F32, KIND_I8_ROWSCALE_F32, make_descs, unpack_noalloc

pytestmark = pytest.mark.gpu


def test_two_tiles_to_a_workgroup():
    n = 4096 * 2064384 + 4097
    rows, cols = 33, 1155
    rng = np.random.default_rng(3)
    q = rng.integers(-127, 128, (rows, cols), dtype=np.int8)
    s = np.exp(rng.normal(-6, 0.5, rows)).astype(np.float32)
    src = torch.empty(2 * n + q.size, dtype=torch.uint8, device="cuda")
    wide = src[:2 * n].view(torch.bfloat16)
    step = 1 << 30
    for at in range(0, n, step):
        m = min(step, n - at)
        wide[at:at + m].copy_(torch.arange(at, at + m, device="cuda", dtype=torch.int64).remainder_(65521).float())
    src[2 * n:].copy_(torch.from_numpy(q.view(np.uint8).reshape(-1)).cuda())
    dst = torch.full((n + q.size + 64,), -7.0, device="cuda")
    unpack_noalloc(make_descs([(KIND_BF16_F32, 0, 0, n // 4097, 4097, 0, 0),
                               (KIND_BF16_F32, 2 * (n // 4097) * 4097, 4 * (n // 4097) * 4097, 1, n % 4097, 0, 0),
                               (KIND_I8_ROWSCALE_F32, 2 * n, 4 * n, rows, cols, 0, 0)]),
                   src, dst, torch.from_numpy(s).cuda())
    for at in range(0, n, step):
        m = min(step, n - at)
        assert torch.equal(dst[at:at + m], wide[at:at + m].float()), at
    np.testing.assert_array_equal(dst[n:n + q.size].cpu().numpy().reshape(rows, cols).view(np.uint32),
                                  oq.dequant_rows(q, s, None, rows, cols, out="float32").view(np.uint32))
    assert bool((dst[n + q.size:] == -7.0).all())
