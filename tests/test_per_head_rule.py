"""Where the waves of a stream workgroup take a head each of whole sequences: the lines of the rule, and what patched
plans keep of it."""
import numpy as np
import pytest

from chunk_attn import capi
from test_tables_native import check_plan


def _tables(lengths, c=64, heads=32, shared=0, **kw):
    tree = capi.Tree(c, sum(n // c + 8 for n in lengths) + shared // c + 2)
    for s, n in enumerate(lengths):
        tree.add_seq(list(range(shared)) + [100_000 * (s + 1) + i for i in range(n)])
    return tree, capi.HostTables(tree.get_chunks(), tree.n_seqs, c, n_heads=heads, **kw)


@pytest.mark.parametrize("lengths,heads,taken", [
    ([2000] * 64, 32, True),             # one round, 333 -> 315 us
    ([2000] * 66, 32, False),            # and a bit, 346 -> 383
    ([4096] * 32, 32, True),             # half of one, 338 -> 323
    ([4096] * 31, 32, False),
    ([2000] * 96, 32, True),             # one and a half, 495 -> 466
    ([2000] * 95, 32, False),
    ([1000] * 64, 32, True), ([999] * 64, 32, False),
    ([2000] * 63 + [1000], 32, True), ([2000] * 50 + [1700] * 14, 32, True), ([1900] * 63 + [2500], 32, False),
    ([3000] * 256, 8, True), ([2000] * 170, 12, True),
    ([2000] * 64, 30, False), ([2000] * 64, 33, False),      # heads that no four share
])
def test_lines_of_the_rule(lengths, heads, taken):
    assert _tables(lengths, heads=heads)[1].plan()["stream_per_head"] == taken


def test_what_else_keeps_the_tiles_in_turn():
    assert not _tables([2000] * 64, shared=64)[1].plan()["stream_per_head"]
    for kw in ({"stream_chunks": 8}, {"partition": 2}, {"partition": 1}):
        assert not _tables([2000] * 64, **kw)[1].plan()["stream_per_head"]
    # chunks that several sequences stream
    assert not _tables([2000] * 64, shared=64, tpp_threshold=100)[1].plan()["stream_per_head"]


@pytest.mark.parametrize("c", [32, 64, 128])
def test_whole_sequences_leave_no_partial_rows_and_grow_with_their_tails(c):
    lengths = [2047 - s % 3 for s in range(64)]
    tree, tables = _tables(lengths, c)
    for step in range(6):
        plan = tables.plan()
        check_plan(tree.get_chunks(), 64, c, plan, 1, 0)
        assert plan["stream_per_head"] and plan["n_part_rows"] == 0 and len(plan["stream_items"]) == 64
        delta = 0
        while not any(f + delta == c for f in plan["tail_fill"]):     # to the step on which last chunks are full
            tree.append_token([90_000_000 + 100 * step + s for s in range(64)])
            delta += 1
        seqs, slots = tree.reserve_tails()
        tables.roll_tails(delta, seqs, slots)
        again = capi.HostTables(tree.get_chunks(), 64, c, n_heads=32, like=tables)
        for key in ("stream_items", "slots", "part_ptr", "seq_len"):
            np.testing.assert_array_equal(np.asarray(tables.plan()[key]), np.asarray(again.plan()[key]))
