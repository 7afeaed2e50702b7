"""Chunk digests and flags at the numbers and sizes of chunks where the launch takes another workgroup
size: fewer chunks than compute units, up to one and a half per unit, more, and long launches of
large chunks; chunks too small for the larger workgroups; a short last chunk in each. Compared with
the host digest (digests and flags are whole numbers, equal bit for bit)."""
from __future__ import annotations

import numpy as np
import pytest

from stagehand_amd import _native
from tests.test_digest import digest_host

pytestmark = pytest.mark.gpu

KIB = 1024


@pytest.mark.parametrize("chunks,chunk", [(1, 64 * KIB), (3, 32 * KIB), (7, 16 * KIB), (255, 64 * KIB), (256, 64 * KIB),
                                          (256, 32 * KIB), (384, 32 * KIB), (385, 32 * KIB), (300, 16 * KIB),
                                          (2, 1024 * KIB), (1792, 256 * KIB), (1793, 256 * KIB)])
def test_digests_and_flags_at_every_workgroup_size(chunks, chunk):
    import torch

    n = (chunks - 1) * chunk + (chunk if chunks % 2 else chunk // 2 + 13)
    g = torch.Generator(device="cuda").manual_seed(chunks)
    dev = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)
    dig = torch.zeros(2 * chunks, dtype=torch.int64, device="cuda")
    flags = torch.full((chunks + 8,), 7, dtype=torch.uint8, pin_memory=True)
    stream = torch.cuda.current_stream().cuda_stream
    _native.call("sh_block_digest", dev.data_ptr(), n, chunk, dig.data_ptr(), stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dig.cpu().numpy().view(np.uint64), digest_host(dev.cpu().numpy(), chunk))
    hit = sorted({0, chunks // 2, chunks - 1})
    for c in hit:
        dev[min(c * chunk + chunk - 1, n - 1)] ^= 1
    _native.call("sh_block_changed", dev.data_ptr(), n, chunk, dig.data_ptr(), flags.data_ptr(), stream)
    torch.cuda.synchronize()
    want = np.zeros(chunks, np.uint8)
    want[hit] = 1
    np.testing.assert_array_equal(flags[:chunks].numpy(), want)
    assert (flags[chunks:] == 7).all()
