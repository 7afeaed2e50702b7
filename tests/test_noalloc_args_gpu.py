"""``sh_unpack_noalloc`` around the limits of a table that travels in the launch's arguments (32
descriptors, 49152 tiles): the same bytes as the plan-based entry point on both sides of them, on two
streams at once and in order across them, and at every replay of a captured call."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from stagehand_amd.unpack import (
    KIND_BF16_F32,
    KIND_COPY_BYTES,
    KIND_F32_BF16,
    KIND_I8_ROWSCALE_BF16,
    KIND_I8_ROWSCALE_F32,
    KIND_ZERO_BYTES,
    UnpackPlan,
    make_descs,
    unpack_noalloc,
)

pytestmark = pytest.mark.gpu

KINDS = [(KIND_I8_ROWSCALE_BF16, 1, 2), (KIND_F32_BF16, 4, 2), (KIND_I8_ROWSCALE_F32, 1, 4), (KIND_BF16_F32, 2, 4),
         (KIND_COPY_BYTES, 1, 1), (KIND_ZERO_BYTES, 0, 1)]


def _table(n: int, kinds=KINDS):
    """n regions of changing kind and size (one element to several tiles); (descs, source bytes,
    destination bytes, scales)."""
    rows, src, dst, scale = [], 3, 0, 0
    for i in range(n):
        kind, ib, ob = kinds[i % len(kinds)]
        r, c = (5 + i, 77 + 613 * (i % 7)) if kind in (KIND_I8_ROWSCALE_BF16, KIND_I8_ROWSCALE_F32) else (1, 1 + 3001 * i)
        dst = -(-dst // ob) * ob
        rows.append((kind, src if ib else 0, dst, r, c, 0, scale))
        src += r * c * ib
        dst += r * c * ob
        scale += r
    return make_descs(rows), src, dst, scale


def _inputs(src_bytes: int, n_scale: int, seed: int):
    g = torch.Generator(device="cuda").manual_seed(seed)
    src = torch.randint(0, 256, (src_bytes + 16,), dtype=torch.uint8, device="cuda", generator=g)
    return src, torch.rand(max(n_scale, 1), device="cuda", generator=g), torch.randn(max(n_scale, 1), device="cuda", generator=g)


def _want(descs, src, dst_bytes, scales, zps):
    want = torch.full((dst_bytes + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    plan = UnpackPlan(descs)
    plan.run(src, want, scales, zps)
    plan.close()
    return want


@pytest.mark.parametrize("n", [1, 2, 7, 31, 32, 33])
@pytest.mark.parametrize("zp", [False, True])
def test_tables_on_both_sides_of_the_argument_limit(n, zp):
    descs, sb, db, ns = _table(n)
    src, scales, zps = _inputs(sb, ns, n)
    want = _want(descs, src, db, scales, zps if zp else None)
    got = torch.full_like(want, 0xA5)
    unpack_noalloc(descs, src, got, scales, zps if zp else None)
    assert torch.equal(got, want)


@pytest.mark.parametrize("tiles", [32768, 32769, 49152, 49153])
def test_tile_limit_of_the_arguments(tiles):
    n = 8192 * tiles
    src = torch.arange(n // 8, device="cuda").view(torch.uint8)
    got = torch.zeros_like(src)
    unpack_noalloc(make_descs([(KIND_COPY_BYTES, 0, 0, 1, n, 0, 0)]), src, got)
    assert torch.equal(got, src)


@pytest.mark.parametrize("zp", [False, True])
def test_long_table_of_several_kinds(zp):
    """More tiles than the arguments take, of aligned int8 rows between a copy and a short odd region."""
    rows, cols = 49160, 8192
    descs = make_descs([(KIND_COPY_BYTES, 0, 0, 1, 1001, 0, 0), (KIND_I8_ROWSCALE_BF16, 1001, 1002, rows, cols, 0, 0),
                        (KIND_I8_ROWSCALE_BF16, 1001 + rows * cols, 1002 + 2 * rows * cols, 7, 333, 0, rows)])
    n_scale = rows + 7
    src, scales, zps = _inputs(1001 + rows * cols + 7 * 333, n_scale, 5)
    dst_bytes = 1002 + 2 * rows * cols + 2 * 7 * 333
    want = _want(descs, src, dst_bytes, scales, zps if zp else None)
    got = torch.full_like(want, 0xA5)
    unpack_noalloc(descs, src, got, scales, zps if zp else None)
    assert torch.equal(got, want)


def test_short_and_long_tables_on_two_streams():
    cases = []
    for n in (32, 40, 3, 64):
        descs, sb, db, ns = _table(n)
        src, scales, _z = _inputs(sb, ns, n)
        cases.append((descs, src, scales, _want(descs, src, db, scales, None)))
    outs = [[torch.full_like(c[3], 0xA5) for c in cases] for _ in range(2)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for i in range(len(cases)):
        for j, stream in enumerate(streams):
            descs, src, scales, _w = cases[(i + j) % len(cases)]
            unpack_noalloc(descs, src, outs[j][(i + j) % len(cases)], scales, stream=stream)
    torch.cuda.synchronize()
    for out in outs:
        for got, case in zip(out, cases):
            assert torch.equal(got, case[3])


@pytest.mark.parametrize("first", [1, 32, 40])
@pytest.mark.parametrize("second", [1, 40])
def test_a_call_waits_for_the_one_before_it_on_another_stream(first, second):
    """The second call reads what the first writes, on a stream of its own and with no other order
    between them than the calls'. The first one's stream is busy for about a millisecond before."""
    n = 40 * 4096
    g = torch.Generator(device="cuda").manual_seed(first + second)
    src = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)
    mid, out = torch.zeros_like(src), torch.zeros_like(src)
    big = torch.zeros(2 << 30, dtype=torch.uint8, device="cuda")
    busy = torch.empty_like(big)

    def copies(regions: int):
        each = n // regions
        sizes = [each] * (regions - 1) + [n - each * (regions - 1)]
        return make_descs([(KIND_COPY_BYTES, each * i, each * i, 1, size, 0, 0) for i, size in enumerate(sizes)])

    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        busy.copy_(big)
    unpack_noalloc(copies(first), src, mid, stream=a)
    unpack_noalloc(copies(second), mid, out, stream=b)
    torch.cuda.synchronize()
    assert torch.equal(out, src)


def test_captured_call_at_every_replay():
    """A captured call with a short table shares nothing with other calls: an eager one with a long
    table (in the scratch array) on a second stream may overlap its replays."""
    descs, sb, db, ns = _table(12)
    src, scales, _z = _inputs(sb, ns, 1)
    got = torch.full((db + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    unpack_noalloc(descs, src, got, scales)  # kernels loaded before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        unpack_noalloc(descs, src, got, scales)
    other, osb, odb, ons = _table(40)
    osrc, oscales, _z = _inputs(osb, ons, 2)
    owant = _want(other, osrc, odb, oscales, None)
    eager = torch.empty_like(owant)
    side = torch.cuda.Stream()
    for seed in range(3, 6):
        src.copy_(_inputs(sb, ns, seed)[0])
        got.fill_(0xA5)
        eager.fill_(0xA5)
        want = _want(descs, src, db, scales, None)
        torch.cuda.synchronize()
        for _ in range(3):
            graph.replay()
            unpack_noalloc(other, osrc, eager, oscales, stream=side)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(eager, owant)
