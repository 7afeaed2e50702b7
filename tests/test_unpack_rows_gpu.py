"""Unpack of rows that are no whole number of chunks and of padded source rows against the CPU oracle
bit for bit, with canary bytes on both sides.

The sizes sit where the kernels' paths meet: rows one element shorter, equal to and longer than a
chunk (8 int8 to bf16, 4 to fp32), rows on both sides of 2 KiB of output (1024 bf16, 512 fp32), chunks
that end exactly at a row's end, a source that ends with the last row's last element, and regions of
one tile and one element more. Scales that make NaNs and infinities lie beside ordinary ones, in
chunks of one row and of two.

Regions just below and above 131072 elements: from there on the tiles of a dequant, cast or widen start
on a destination boundary whatever the region's start, and its first chunk is cut."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import squareq as oq
from stagehand_amd.unpack import (
    KIND_BF16_F32,
    KIND_COPY_BYTES,
    KIND_F32_BF16,
    KIND_I8_ROWSCALE_BF16,
    KIND_I8_ROWSCALE_F32,
    KIND_ZERO_BYTES,
    UnpackPlan,
    make_descs,
)

pytestmark = pytest.mark.gpu

ROWS = [
    # rows, cols, padding of a source row
    (300, 1, 0), (300, 1, 3), (200, 3, 1), (200, 4, 0), (200, 4, 5), (200, 5, 3), (90, 7, 2), (90, 8, 0), (90, 8, 8),
    (90, 9, 0), (90, 9, 7), (33, 1155, 0), (33, 1155, 16), (5, 4097, 1), (2, 8193, 0),
    (64, 2048, 16), (128, 1023, 0), (128, 1024, 0), (128, 1025, 3), (43, 3072, 0), (43, 3072, 4),
    # the line between narrow and wide rows (2 KiB of output), and narrow rows of whole chunks in regions
    # long enough to start on a boundary from any element, so that their chunks cross rows
    (300, 511, 0), (300, 512, 0), (300, 513, 0), (2100, 64, 0), (8200, 16, 0), (16400, 8, 0), (32800, 4, 0), (160, 1016, 0),
    (257, 511, 1),
]


def _dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("rows,cols,pad", ROWS)
@pytest.mark.parametrize("out", ["bfloat16", "float32"])
@pytest.mark.parametrize("start,zp", [(0, False), (1, True), (5, False), (8, True), (2047, False)])
def test_rows_of_any_length_stride_and_start(rows, cols, pad, out, start, zp):
    rng = np.random.default_rng(rows * 131 + cols * 7 + pad + start)
    ld = cols + pad
    src_off = start % 7
    src = np.full(src_off + (rows - 1) * ld + cols, 99, np.uint8)  # the last row's padding is not there
    q = rng.integers(-128, 128, (rows, ld), dtype=np.int8)
    src[src_off:] = q.view(np.uint8).reshape(-1)[:(rows - 1) * ld + cols]
    s = np.exp(rng.normal(-6.0, 0.5, rows + 2)).astype(np.float32)
    s[2::5] = np.array([np.inf, np.nan, -1.5, 1e-42], np.float32)[np.arange(s[2::5].size) % 4]
    z = rng.normal(0, 3, rows + 2).astype(np.float32) if zp else None
    width, kind = (2, KIND_I8_ROWSCALE_BF16) if out == "bfloat16" else (4, KIND_I8_ROWSCALE_F32)
    dst_off = 4096 + width * start
    dst = torch.full((dst_off + rows * cols * width + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
    UnpackPlan(make_descs([(kind, src_off, dst_off, rows, cols, ld, 2)])).run(
        _dev(src), dst, _dev(s), _dev(z) if zp else None)
    got = dst.cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        want = oq.dequant_rows(q, s[2:], z[2:] if zp else None, rows, cols, out=out)
    body = got[dst_off:dst_off + rows * cols * width]
    if width == 2:
        np.testing.assert_array_equal(body.view(np.uint16).reshape(rows, cols), want)
    else:  # a NaN's payload is not defined for fp32 arithmetic
        body, want = body.view(np.float32).reshape(rows, cols), want
        np.testing.assert_array_equal(np.isnan(body), np.isnan(want))
        np.testing.assert_array_equal(np.where(np.isnan(body), 0, body).view(np.uint32),
                                      np.where(np.isnan(want), 0, want).view(np.uint32))
    assert (got[:dst_off] == 0xAB).all() and (got[dst_off + rows * cols * width:] == 0xAB).all()


@pytest.mark.parametrize("numel", [1, 5, 8193, (1 << 17) - 1, 1 << 17, (1 << 17) + 4099])
@pytest.mark.parametrize("start", [0, 1, 3, 16, 2047])
def test_flat_regions_from_any_start(numel, start):
    """Every flat kind in one plan, each region ``start`` elements past a 4 KiB boundary."""
    rng = np.random.default_rng(numel + start)
    f = rng.normal(0, 1, numel).astype(np.float32)
    bf = oq.cast_f32_bf16(rng.normal(0, 1, numel).astype(np.float32))
    raw = rng.integers(0, 256, numel, dtype=np.uint8)
    parts = [f.view(np.uint8), bf.view(np.uint8), raw]
    src = np.concatenate([np.zeros(3, np.uint8)] + parts)
    at = np.cumsum([3] + [p.size for p in parts])
    kinds = [(KIND_F32_BF16, 2), (KIND_BF16_F32, 4), (KIND_COPY_BYTES, 1), (KIND_ZERO_BYTES, 1)]
    descs, spans, pos = [], [], 0
    for i, (kind, width) in enumerate(kinds):
        pos = -(-pos // 4096) * 4096 + width * start
        descs.append((kind, int(at[i]) if i < 3 else 0, pos, 1, numel, 0, 0))
        spans.append((pos, pos + width * numel))
        pos += width * numel
    dst = torch.full((pos + 4096,), 0xAB, dtype=torch.uint8, device="cuda")
    UnpackPlan(make_descs(descs)).run(_dev(src), dst)
    got = dst.cpu().numpy()
    body = [got[a:b] for a, b in spans]
    np.testing.assert_array_equal(body[0].view(np.uint16), oq.cast_f32_bf16(f))
    np.testing.assert_array_equal(body[1].view(np.float32), oq.bf16_bits_to_f32(bf))
    np.testing.assert_array_equal(body[2], raw)
    assert not body[3].any()
    outside = np.ones(got.size, bool)
    for a, b in spans:
        outside[a:b] = False
    assert (got[outside] == 0xAB).all()


@pytest.mark.parametrize("numel", [2048 * 32768, 2048 * 32768 + 1])
def test_cast_of_whole_tiles_and_one_element_more(numel):
    """A cast-only plan of whole tiles of 2048 elements and of one element more; torch's device cast rounds
    the same way (no NaN here)."""
    g = torch.Generator(device="cuda").manual_seed(numel)
    src = torch.randn(numel, device="cuda", generator=g)
    dst = torch.empty(numel, dtype=torch.bfloat16, device="cuda")
    plan = UnpackPlan(make_descs([(KIND_F32_BF16, 0, 0, 1, numel, 0, 0)]))
    assert plan.info["n_tiles"] == -(-numel // 2048)
    plan.run(src, dst)
    assert torch.equal(dst, src.to(torch.bfloat16))
