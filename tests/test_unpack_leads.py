"""Where a plan's tiles start in a region whose destination is no whole number of chunks past a 4 KiB
boundary (CPU only: ``sh_plan_describe``). From 131072 elements on, the lead of a dequant, cast or widen
before element 0 reaches back to the boundary all the same; shorter regions and the other kinds (a
byte copy is slower so) get none."""
from __future__ import annotations

import numpy as np
import pytest

from stagehand_amd import _native
from stagehand_amd._native import PLAN_INFO_DTYPE
from stagehand_amd.unpack import (
    KIND_BF16_F32,
    KIND_COPY_BYTES,
    KIND_F32_BF16,
    KIND_I8_ROWSCALE_BF16,
    KIND_I8_ROWSCALE_F32,
    KIND_ZERO_BYTES,
    make_descs,
)

MIN_LEAD = 1 << 17
# kind: (elements per tile, bytes of an output element)
KINDS = {KIND_I8_ROWSCALE_BF16: (8192, 2), KIND_I8_ROWSCALE_F32: (4096, 4), KIND_F32_BF16: (2048, 2),
         KIND_BF16_F32: (4096, 4)}
NO_LEAD = {KIND_COPY_BYTES: (8192, 1), KIND_ZERO_BYTES: (16384, 1)}


def tiles(kind: int, dst_off: int, cols: int, rows: int = 1) -> int:
    table = make_descs([(kind, 0, dst_off, rows, cols, 0, 0)])
    info = np.zeros(1, dtype=PLAN_INFO_DTYPE)
    _native.call("sh_plan_describe", table.ctypes.data, 1, info.ctypes.data)
    return int(info[0]["n_tiles"])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("lead", [1, 3, 5, 1021])
def test_a_long_region_gets_a_lead_of_any_length(kind, lead):
    per_tile, width = KINDS[kind]
    for numel in (MIN_LEAD, MIN_LEAD + per_tile - lead, MIN_LEAD + per_tile - lead + 1):
        assert tiles(kind, 4096 + lead * width, numel) == -(-(numel + lead) // per_tile), numel
        # a start inside an element's worth of bytes: no lead reaches the boundary
        assert tiles(kind, 4096 + lead * width + 1, numel) == -(-numel // per_tile)
    short = MIN_LEAD - 1 - (MIN_LEAD - 1) % per_tile  # whole tiles, below the line
    assert tiles(kind, 4096 + lead * width, short) == short // per_tile


@pytest.mark.parametrize("kind", NO_LEAD)
def test_the_other_kinds_get_whole_chunk_leads_only(kind):
    per_tile, width = NO_LEAD[kind]
    for lead in (1, 3, 5, 1021):
        assert tiles(kind, 4096 + lead * width, 64 * per_tile) == 64, lead


def test_a_ragged_lead_never_refuses_a_table_that_fits_without_it():
    """The largest launch holds (2^32 - 1) // 512 tiles, the allocation-free table 2064384: a region of
    exactly that many stays accepted from a start whose lead, no whole number of chunks, would add one.
    A lead of whole chunks is part of every form of a table: it adds a tile to each of the region's 16
    pieces of 2^30 elements."""
    max_tiles = (2**32 - 1) // 512
    assert tiles(KIND_F32_BF16, 4096 + 2, 2048, rows=max_tiles) == max_tiles
    with pytest.raises(ValueError, match="tiles"):
        tiles(KIND_F32_BF16, 4096 + 64, 2048, rows=max_tiles)
    assert tiles(KIND_F32_BF16, 4096 + 64, 2048, rows=max_tiles - 16) == max_tiles
    lib = _native.lib()
    for rows, message in ((2064384, b"source"), (2064385, b"tiles")):  # fits: refused for its buffers alone
        table = make_descs([(KIND_F32_BF16, 0, 4098, rows, 2048, 0, 0)])
        assert lib.sh_unpack_noalloc(table.ctypes.data, 1, None, 0, None, None, 0, None, 0,
                                     None) == _native.SH_ERR_INVALID
        assert message in lib.sh_last_error()


def test_fp32_outputs_near_the_launch_limit_take_two_tiles_to_a_workgroup():
    """A tile of an fp32 output is 4096 elements. A table of more tiles than a launch holds is built with
    two to a workgroup, so that regions of up to 8192 elements per workgroup are accepted."""
    max_tiles = (2**32 - 1) // 512
    for kind in (KIND_I8_ROWSCALE_F32, KIND_BF16_F32):
        assert tiles(kind, 0, 4096, rows=max_tiles) == max_tiles
        assert tiles(kind, 0, 8192, rows=max_tiles) == max_tiles
        with pytest.raises(ValueError, match="tiles"):
            tiles(kind, 0, 8192, rows=max_tiles + 1)
    lib = _native.lib()
    for rows, message in ((2064384, b"source"), (2064385, b"tiles")):
        table = make_descs([(KIND_BF16_F32, 0, 0, rows, 8192, 0, 0)])
        assert lib.sh_unpack_noalloc(table.ctypes.data, 1, None, 0, None, None, 0, None, 0,
                                     None) == _native.SH_ERR_INVALID
        assert message in lib.sh_last_error()
