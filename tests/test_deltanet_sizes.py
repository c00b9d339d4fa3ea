"""Which delta-rule calls take the chunk form, and its scratch (host arithmetic, no device call)."""

from __future__ import annotations

import pytest

import _mtpk


@pytest.fixture(scope="module")
def need():
    if not _mtpk.LIB_PATH.exists():
        import __graft_entry__

        __graft_entry__.build()
    fn = _mtpk.lib().mtpk_delta_rule_workspace_bytes
    return lambda rows, t, out, heads=64, qk=16, kd=128, vd=128: fn(rows, t, heads, qk, kd, vd, int(out))


@pytest.mark.parametrize("rows,t,out,heads", [
    # measured with 64 heads of 128 x 128, step by step / chunks in us: 24 / 29, 36 / 42, 57 / 68, 108 / 113,
    # 82 / 94, 82 / 116, 107 / 118, 209 / 248, 184 / 273, 130 / 208, 643 / 785
    (1, 16, True, 64), (2, 24, True, 64), (4, 32, True, 64), (4, 65, True, 64), (6, 48, True, 64), (8, 48, True, 64),
    (8, 64, True, 64), (8, 129, True, 64), (12, 96, True, 64), (16, 64, True, 64), (16, 320, True, 64),
    # commits: 26 / 31 (launches), 81 / 87, 77 / 74 (within what runs differ), and rows that fill the chip
    (1, 20, False, 64), (8, 64, False, 64), (8, 65, False, 64), (32, 128, False, 64),
    (1, 16, True, 4), (1, 20, False, 4),  # few heads: the launches
    (64, 15, True, 64), (1, 15, True, 64), (1, 1, False, 64),
])
def test_calls_that_stay_step_by_step(need, rows, t, out, heads) -> None:
    assert need(rows, t, out, heads, min(heads, 16)) == 0


@pytest.mark.parametrize("rows,t,out,heads", [
    # 35 / 29, 57 / 44, 68 / 56, 82 / 68, 106 / 95, 107 / 69, 207 / 116, 400 / 314, 2286 / 178
    (1, 24, True, 64), (2, 40, True, 64), (3, 40, True, 64), (4, 48, True, 64), (6, 64, True, 64), (4, 64, True, 64), (4, 128, True, 64), (8, 256, True, 64), (1, 1500, True, 64),
    # 34 / 25, 42 / 33, 76 / 51, 149 / 131, 1637 / 116
    (1, 32, False, 64), (2, 40, False, 64), (4, 64, False, 64), (8, 128, False, 64), (1, 1500, False, 64),
    (1, 24, True, 4), (1, 32, False, 4),
])
def test_calls_that_take_the_chunks(need, rows, t, out, heads) -> None:
    assert need(rows, t, out, heads, min(heads, 16)) > 0


def test_shapes_the_chunk_form_does_not_have(need) -> None:
    assert need(1, 1500, True, kd=64) == need(1, 1500, True, vd=96) == need(1, 1500, True, qk=5) == 0
    assert need(1, 65600, True) == 0  # 32-bit offsets inside a row


@pytest.mark.parametrize("out", [True, False])
def test_scratch_of_long_rows_is_bounded(need, out) -> None:
    """57 KB a step of 64 heads with outputs: a long row goes in pieces, more rows in groups."""
    assert all(0 < need(1, t, out) <= 256 << 20 for t in (1500, 4608, 4609, 8192, 32768, 65000))
    assert need(1, 1500, out) < need(4, 1500, out) <= 256 << 20
    assert need(1, 64, out) < need(1, 65, out)
