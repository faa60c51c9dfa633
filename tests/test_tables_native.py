"""Device-table flattening (host side of ca_refresh_kernel_context): reference-form tables
bit-exact against the oracle and the hand-worked example; structural invariants of the packed
work list the kernels consume."""
import random

import numpy as np
import pytest

import synth
from chunk_attn import capi
from oracle.prefix_tree import PrefixTree, build_ref_tables
from kats import ADD_SEQ_STEPS, TABLE_KAT


def rows_np(tree: PrefixTree):
    return np.array([r.as_tuple() for r in tree.get_chunks()], np.int32).reshape(-1, 4)


def assert_ref_equal(ref: dict, want):
    assert ref["n_shared"] == want.n_shared
    assert ref["partial_rows"] == want.partial_rows
    assert ref["max_seq_n_chunks"] == want.max_seq_n_chunks
    np.testing.assert_array_equal(ref["final_idx"], want.final_idx)
    np.testing.assert_array_equal(ref["slots"], want.slots)
    np.testing.assert_array_equal(ref["begins"], want.begins)
    np.testing.assert_array_equal(ref["ends"], want.ends)
    np.testing.assert_array_equal(ref["offsets"], want.offsets)
    np.testing.assert_array_equal(ref["seq_n_tokens"], want.seq_n_tokens)
    np.testing.assert_array_equal(ref["seq_chunk_map"], np.array(want.seq_chunk_map, np.int32).reshape(
        ref["seq_chunk_map"].shape))


def test_table_kat():
    t = PrefixTree(2, 64)
    for tokens, _, _ in ADD_SEQ_STEPS:
        t.add_seq(tokens)
    tabs = capi.build_tables(rows_np(t), t.n_seqs, 2, 1)["ref"]
    for key in ("final_idx", "begins", "ends", "offsets", "seq_n_tokens"):
        assert tabs[key].tolist() == TABLE_KAT[key]
    assert tabs["seq_chunk_map"].tolist() == TABLE_KAT["seq_chunk_map"]
    assert (tabs["n_shared"], tabs["partial_rows"], tabs["max_seq_n_chunks"]) == (2, 9, 3)


def check_plan(rows, n_seqs, c, plan, tpp, partition):
    """Every (sequence, chunk) pair is attended exactly once, in path order; partial lists
    name exactly the rows the items write."""
    covered = {s: [] for s in range(n_seqs)}        # s -> list of (pos, slot)
    written = {}                                    # absolute part row -> seq
    slots = plan["slots"]
    pp = plan["part_ptr"]
    for it in plan["shared_items"]:
        b, n, sf, nc, pr, pos0, len0, _ = it.tolist()[:8]
        assert 1 <= n <= (128 if it[7] & 1 else 32) and nc >= 1 and pr >= 0
        assert len0 == plan["seq_len"][b] and it[8:8 + min(nc, 8)].tolist() == slots[sf:sf + min(nc, 8)].tolist()
        for i in range(n):
            row = int(pp[b + i]) + pr
            assert row not in written
            written[row] = b + i
            for k in range(nc):
                covered[b + i].append((pos0 + k, int(slots[sf + k])))
    for it in plan["stream_items"]:
        s, n, sf, nc, pr, pos0, len0, _ = it.tolist()[:8]
        assert n == 1 and len0 == plan["seq_len"][s] and nc >= 1
        assert it[8:8 + min(nc, 8)].tolist() == slots[sf:sf + min(nc, 8)].tolist()
        if pr >= 0:
            row = int(pp[s]) + pr
            assert row not in written
            written[row] = s
        for k in range(nc):
            covered[s].append((pos0 + k, int(slots[sf + k])))
    # expected coverage from the rows
    want = {s: [] for s in range(n_seqs)}
    depth = [0] * n_seqs
    for (slot, nt, b, e) in rows.tolist():
        for s in range(b, e):
            want[s].append((depth[s], slot))
            depth[s] += 1
    for s in range(n_seqs):
        assert sorted(covered[s]) == want[s]
        lst = list(range(int(pp[s]), int(pp[s + 1])))       # the rows the merge reads
        mine = sorted(r for r, q in written.items() if q == s)
        direct = [it for it in plan["stream_items"] if it[0] == s and it[4] < 0]
        if direct:
            assert lst == [] and mine == [] and len(direct) == 1
        else:
            assert lst == mine and len(mine) >= 1
        assert plan["seq_len"][s] == sum(nt for (_, nt, b, e) in rows.tolist() if b <= s < e)
        last = [r for r in rows.tolist() if r[2] <= s < r[3]][-1]
        assert (plan["tail_slot"][s], plan["tail_fill"][s]) == (last[0], last[1])
    assert all(0 <= r < plan["n_part_rows"] for r in written)
    assert plan["n_part_rows"] == int(pp[n_seqs]) == len(written)
    if partition == 2:
        assert len(plan["shared_items"]) == 0
    if partition == 1:
        assert len(plan["stream_items"]) == 0
    if partition == 0:
        for it in plan["shared_items"]:
            pass
        shared_rows = rows[(rows[:, 3] - rows[:, 2]) > tpp]
        assert plan["shared_tokens"] == int(shared_rows[:, 1].sum())


@pytest.mark.parametrize("seed", range(8))
def test_random_trees(seed):
    rng = random.Random(seed)
    c = rng.choice([2, 4])
    t = PrefixTree(c, 4096)
    n = 0
    for _ in range(60):
        op = rng.random()
        if op < 0.6 or n == 0:
            t.add_seq([rng.randint(0, 1) for _ in range(rng.randint(1, 4 * c))])
            n += 1
        elif op < 0.85:
            t.append_token([rng.randint(0, 1) for _ in range(n)])
        else:
            t.remove_seq(rng.randrange(n))
            n -= 1
    rows = rows_np(t)
    for tpp in (0, 1, 2):
        for partition in (0, 1, 2):
            for seg, strm in ((0, 0), (1, 1), (3, 2)):
                out = capi.build_tables(rows, t.n_seqs, c, tpp, partition, seg, strm, n_heads=4, n_cus=8)
                assert_ref_equal(out["ref"], build_ref_tables(rows.tolist(), t.n_seqs, c, tpp))
                check_plan(rows, t.n_seqs, c, out["plan"], tpp, partition)


@pytest.mark.parametrize("cfg", [0, 1, 3])
def test_benchmark_plans(cfg):
    w = synth.baseline_config(cfg)
    need = sum(w.seq_len(s) // w.chunk_size + 2 for s in range(w.n_seqs))
    t = PrefixTree(w.chunk_size, need)
    for s in range(w.n_seqs):
        t.add_seq(w.tokens(s))
    rows = rows_np(t)
    out = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0)
    assert_ref_equal(out["ref"], build_ref_tables(rows.tolist(), t.n_seqs, w.chunk_size, 1))
    check_plan(rows, t.n_seqs, w.chunk_size, out["plan"], 1, 0)
    assert out["plan"]["shared_tokens"] == w.shared_tokens_physical()
    assert out["plan"]["stream_tokens"] == w.logical_tokens() - w.n_seqs * sum(
        len(seg.ids) for seg in w.seqs[0] if seg.k_stream < synth.STREAM_K_UNIQUE)


def test_bad_rows_rejected():
    rows = np.array([[0, 2, 0, 3]], np.int32)
    with pytest.raises(capi.ChunkAttnError):
        capi.build_tables(rows, 2, 2)          # range exceeds n_seqs
    with pytest.raises(capi.ChunkAttnError):
        capi.build_tables(rows, 3, 2, partition=5)


@pytest.mark.parametrize("partition", [0, 1, 2])
@pytest.mark.parametrize("seg,strm", [(0, 0), (500, 500), (64, 63), (65, 64)])
def test_items_never_hold_more_than_64_chunks(partition, seg, strm):
    """The kernels keep an item's slot ids in one register per wave (64 lanes): whatever segment
    or stream sizes are asked for, no work item may exceed 64 chunks, and all chunks are still
    covered exactly once."""
    c = 2
    t = PrefixTree(c, 4096)
    shared = list(range(2 * 150))                 # 150 shared chunks on one path
    for s in range(5):
        t.add_seq(shared + [1000 * (s + 1) + i for i in range(2 * 140 + 1)])   # 141 private chunks each
    rows = rows_np(t)
    out = capi.build_tables(rows, t.n_seqs, c, 1, partition, seg, strm, n_heads=4, n_cus=8)
    plan = out["plan"]
    check_plan(rows, t.n_seqs, c, plan, 1, partition)
    for items in (plan["shared_items"], plan["stream_items"]):
        if len(items):
            assert items[:, 3].min() >= 1 and items[:, 3].max() <= 64


def test_stream_items_taper_over_the_last_sequences():
    """With the default item size, the last sequences (one fill of the device's workgroup slots,
    or a quarter of the sequences if that is more, at most half) get items of half the length:
    the launch drains through them.  An explicit item size switches the taper off, and sizes
    that cannot be halved (half an item would leave waves without a tile) stay as they are."""
    w = synth.baseline_config(1)                      # 32 sequences, 8 private chunks of 64 (+ empty tail) each
    t = PrefixTree(w.chunk_size, 2048)
    for s in range(w.n_seqs):
        t.add_seq(w.tokens(s))
    rows = rows_np(t)
    plan = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0)["plan"]
    check_plan(rows, t.n_seqs, w.chunk_size, plan, 1, 0)
    per_seq = np.bincount(plan["stream_items"][:, 0], minlength=w.n_seqs)
    # 256 compute units x 2 slots / 32 heads = 16 sequences per fill = half of the 32: the cap
    assert per_seq[:16].tolist() == [1] * 16 and per_seq[16:].tolist() == [2] * 16
    assert plan["stream_items"][:16, 3].tolist() == [9] * 16            # 8 chunks and the tail riding along
    assert sorted(set(plan["stream_items"][16:, 3].tolist())) == [4, 5]
    small = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0, n_heads=32, n_cus=64)["plan"]   # 4 per fill
    assert np.bincount(small["stream_items"][:, 0], minlength=w.n_seqs).tolist() == [1] * 24 + [2] * 8   # a quarter
    fixed = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0, 0, 8)["plan"]
    assert np.bincount(fixed["stream_items"][:, 0], minlength=w.n_seqs).tolist() == [1] * 32
    # chunk size 128: the default item is four chunks, one per wave: no taper
    t2 = PrefixTree(128, 2048)
    for s in range(16):
        t2.add_seq(list(range(256)) + [10 ** 6 * (s + 1) + i for i in range(8 * 128)])
    p2 = capi.build_tables(rows_np(t2), 16, 128, 1, 0)["plan"]
    assert len(set(np.bincount(p2["stream_items"][:, 0], minlength=16).tolist())) == 1


def test_shared_runs_of_different_widths_get_segments_of_similar_cost():
    """Two-level workload: the root run (64 sequences, two 32-row items per segment, 16 chunks)
    costs more per tile than the eight group runs (8 sequences, 8 chunks each), which are the
    majority of the chunk-first workgroups; the root is cut into three segments instead of two so
    that no chunk-first workgroup outlasts the others by much.  Single-run workloads keep their
    segmentation, and an explicit segment length switches the balancing off."""
    w = synth.baseline_config(3)
    t = PrefixTree(w.chunk_size, 2048)
    for s in range(w.n_seqs):
        t.add_seq(w.tokens(s))
    rows = rows_np(t)
    plan = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0)["plan"]
    check_plan(rows, t.n_seqs, w.chunk_size, plan, 1, 0)
    items = plan["shared_items"]
    root = items[items[:, 1] == 32]                    # 32-row items: the root run, two per segment
    mid = items[items[:, 1] == 8]
    assert len(root) == 6 and sorted(root[:, 3].tolist()) == [5, 5, 5, 5, 6, 6]
    assert len(mid) == 8 and set(mid[:, 3].tolist()) == {8}
    fixed = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0, 8, 0)["plan"]["shared_items"]
    assert len(fixed[fixed[:, 1] == 32]) == 4
    w2 = synth.baseline_config(1)                      # one shared run: nothing to balance against
    t2 = PrefixTree(w2.chunk_size, 2048)
    for s in range(w2.n_seqs):
        t2.add_seq(w2.tokens(s))
    assert len(capi.build_tables(rows_np(t2), t2.n_seqs, w2.chunk_size, 1, 0)["plan"]["shared_items"]) == 2


def test_wide_form_for_33_to_95_sequences_needs_a_long_run():
    """Chunks covering 96 sequences or more always take the row-split wide form (flag 1, one item
    of up to 128 rows per segment).  From 33 to 95 sequences (more than one 32-row item) they take
    it when their run holds at least 2048 tokens; shorter runs, and anything up to 32 sequences,
    stay with 32-row items."""
    def shared_items(n_seqs, shared_chunks, c=64):
        t = PrefixTree(c, 8192)
        prefix = list(range(shared_chunks * c))
        for s in range(n_seqs):
            t.add_seq(prefix + [10 ** 6 * (s + 1) + i for i in range(c)])
        rows = rows_np(t)
        plan = capi.build_tables(rows, t.n_seqs, c, 1, 0)["plan"]
        check_plan(rows, t.n_seqs, c, plan, 1, 0)
        return plan["shared_items"]

    for n_seqs, chunks, wide in ((64, 32, True), (64, 31, False), (64, 16, False), (95, 32, True),
                                 (63, 64, True), (33, 32, True), (33, 31, False), (32, 64, False),
                                 (96, 4, True), (130, 4, True)):
        items = shared_items(n_seqs, chunks)
        assert set(items[:, 7].tolist()) == {1 if wide else 0}, (n_seqs, chunks)
        assert items[:, 1].max() == (min(n_seqs, 128) if wide else 32), (n_seqs, chunks)
    # chunk size 32: the same 2048 tokens are 64 chunks
    assert set(shared_items(64, 64, c=32)[:, 7].tolist()) == {1}
    assert set(shared_items(64, 63, c=32)[:, 7].tolist()) == {0}


def test_all_shared_wide_runs_get_one_workgroup_per_compute_unit():
    """Sharing sweep at fraction 1.0 (64 sequences share all 64 chunks, nothing private): the step is
    short, so the shared run is cut until its workgroups fit the device in one go, and a wide
    workgroup counts for two slots: 8 segments of 8 chunks x 32 heads = 256 workgroups on 256
    compute units.  With long private parts (fraction 0.75) the run stays in one piece."""
    def plan_for(fraction, **kw):
        w = synth.baseline_config(2, fraction=fraction)
        t = PrefixTree(w.chunk_size, 8192)
        for s in range(w.n_seqs):
            t.add_seq(w.tokens(s))
        rows = rows_np(t)
        plan = capi.build_tables(rows, t.n_seqs, w.chunk_size, 1, 0, **kw)["plan"]
        check_plan(rows, t.n_seqs, w.chunk_size, plan, 1, 0)
        return plan["shared_items"]
    items = plan_for(1.0)
    assert len(items) == 8 and set(items[:, 3].tolist()) == {8} and set(items[:, 7].tolist()) == {1}
    assert set(items[:, 1].tolist()) == {64}
    half = plan_for(1.0, n_heads=32, n_cus=128)            # half the device: twice the segment length
    assert len(half) == 4 and set(half[:, 3].tolist()) == {16}
    long_private = plan_for(0.75)
    assert len(long_private) == 1 and long_private[0, 3] == 48 and long_private[0, 7] == 1


def assert_plans_equal(a: dict, b: dict):
    assert sorted(a) == sorted(b)
    for key in a:
        if isinstance(a[key], np.ndarray):
            np.testing.assert_array_equal(a[key], b[key], err_msg=key)
        else:
            assert a[key] == b[key], key


@pytest.mark.parametrize("seed", range(10))
def test_rolled_tables_equal_rebuilt_tables(seed):
    """Decode steps on a random tree: whenever last chunks fill up, the tables patched in place
    (ca_tables_roll_tails, the host half of ca_ctx_roll_tails) equal the tables built from a walk
    of the tree in its new state with the same work-item sizes."""
    rng = random.Random(100 + seed)
    c = rng.choice([2, 4, 64])
    partition = rng.choice([0, 0, 2])
    tpp = rng.choice([1, 1, 2])
    tree = capi.Tree(c, 4096)
    fams = [[rng.randint(0, 3) for _ in range(rng.randint(c, 6 * c))] for _ in range(3)]
    n = rng.randint(2, 12)
    for s in range(n):
        f = rng.choice(fams)
        tree.add_seq(f[:rng.randint(1, len(f))] + [100 + 1000 * s + j for j in range(rng.randint(0, 3 * c))])
    kw = dict(n_heads=rng.choice([2, 32]), n_cus=rng.choice([4, 256]))
    first = capi.HostTables(tree.get_chunks(), n, c, tpp, partition, rng.choice([0, 0, 2]), rng.choice([0, 0, 3]), **kw)
    live = capi.HostTables(tree.get_chunks(), n, like=first)
    assert_plans_equal(live.plan(), first.plan())
    delta, rolls = 0, 0
    for step in range(3 * c + 5):
        seqs, slots = tree.reserve_tails()
        if seqs or step % 7 == 3:            # also: fold the appended tokens in with nothing rolled
            live.roll_tails(delta, seqs, slots)
            delta = 0
            rolls += len(seqs)
            rebuilt = capi.HostTables(tree.get_chunks(), n, like=first)
            assert_plans_equal(live.plan(), rebuilt.plan())
            check_plan(tree.get_chunks(), n, c, live.plan(), tpp, partition)
        tree.append_token([5000 + step * 64 + s for s in range(n)])
        delta += 1
    assert rolls >= n


def test_roll_tails_rejects_what_it_cannot_patch():
    c = 4
    tree = capi.Tree(c, 64)
    tree.add_seq([1, 2, 3, 4, 5, 6])
    tree.add_seq([1, 2, 3, 4, 7])
    rows = tree.get_chunks()
    t = capi.HostTables(rows, 2, c)
    before = t.plan()
    with pytest.raises(capi.ChunkAttnError):      # the last chunk of sequence 0 holds 2 of 4 tokens
        t.roll_tails(0, [0], [9])
    with pytest.raises(capi.ChunkAttnError):      # three more tokens do not fit sequence 0's last chunk
        t.roll_tails(3, [], [])
    with pytest.raises(capi.ChunkAttnError):
        t.roll_tails(2, [0, 0], [9, 10])
    with pytest.raises(capi.ChunkAttnError):
        t.roll_tails(2, [5], [9])
    assert_plans_equal(t.plan(), before)
    t.roll_tails(2, [0], [9])                     # sequence 0 full after two tokens: fine
    assert t.plan()["tail_slot"].tolist()[0] == 9 and t.plan()["tail_fill"].tolist() == [0, 3]
    every_chunk_first = capi.HostTables(rows, 2, c, 1, 1)
    with pytest.raises(capi.ChunkAttnError):
        every_chunk_first.roll_tails(2, [0], [9])
    last_chunks_shared = capi.HostTables(rows, 2, c, 0, 0)   # tpp_threshold 0: every chunk is attended chunk-first
    with pytest.raises(capi.ChunkAttnError):
        last_chunks_shared.roll_tails(2, [0], [9])
    # a full last chunk that two sequences stream (rows by hand: the tree keeps last chunks private):
    # where the successors go among the rows is not the patch's to decide
    shared_tail = np.array([[0, 4, 0, 2]], np.int32)
    for kw in ({"partition": 2}, {"tpp_threshold": 2}):
        t2 = capi.HostTables(shared_tail, 2, c, **kw)
        before2 = t2.plan()
        with pytest.raises(capi.ChunkAttnError):
            t2.roll_tails(0, [0, 1], [5, 6])
        assert_plans_equal(t2.plan(), before2)


@pytest.mark.parametrize("cfg,steps", [(0, 1024), (1, 2048), (3, 1024)])
def test_replanning_policy_keeps_patched_tables_near_fresh_ones(cfg, steps):
    """A long decode, tables patched at every roll-over (ca_tables_roll_tails) and rebuilt whenever
    the policy says so (ca_tables_stale, threshold 25 %: what ca_ctx_roll_tails does on the device
    side).  `stale` is exactly "the attended tokens moved by more than 25 % since the last full
    build", and while it is false the patched plan has within 10 % of the work items of a plan built
    afresh from the tree (patch-only drifts to 39 % on the 16-sequence configuration) -- except right
    after the fresh plan has moved to the next length of stream items (they double with the size of
    the step), where the patched one is one doubling behind until the next rebuild."""
    w = synth.baseline_config(cfg)
    c, n = w.chunk_size, w.n_seqs
    tree = capi.Tree(c, 1 << 16)
    for s in range(n):
        tree.add_seq(w.tokens(s))
    live = capi.HostTables(tree.get_chunks(), n, c, n_heads=w.n_heads)
    never = capi.HostTables(tree.get_chunks(), n, c, n_heads=w.n_heads)   # patch-only, for comparison
    built = live.info().shared_tokens + live.info().stream_tokens
    delta, rebuilds, worst, worst_never, one_doubling_behind = 0, 0, 0.0, 0.0, 0
    for step in range(steps):
        seqs, slots = tree.reserve_tails()
        if seqs:
            live.roll_tails(delta, seqs, slots)
            never.roll_tails(delta, seqs, slots)
            delta = 0
            now = live.info().shared_tokens + live.info().stream_tokens
            assert live.stale(25) == (abs(now - built) * 100 > 25 * built)
            assert not live.stale(0) and not never.stale(0)          # 0 switches the policy off
            fresh = capi.HostTables(tree.get_chunks(), n, c, n_heads=w.n_heads)
            n_fresh = fresh.info().n_shared_items + fresh.info().n_stream_items
            worst_never = max(worst_never, abs(never.info().n_shared_items + never.info().n_stream_items - n_fresh) / n_fresh)
            if live.stale(25):
                live, built, rebuilds = fresh, now, rebuilds + 1
                assert not live.stale(25)
            else:
                # the length of a stream item moves in powers of two with the size of the step: where a
                # fresh plan has just taken the next one, the patched plan is one doubling behind
                cut_live = int(live.plan()["stream_items"][:, 3].max())
                cut_fresh = int(fresh.plan()["stream_items"][:, 3].max())
                if abs(cut_live - cut_fresh) <= 1:
                    worst = max(worst, abs(live.info().n_shared_items + live.info().n_stream_items - n_fresh) / n_fresh)
                else:
                    assert cut_fresh / 2.2 <= cut_live <= cut_fresh * 2.2
                    one_doubling_behind += 1
        else:
            # tokens appended since the last patch count as well when the caller passes them
            assert live.stale(25, delta * n) == (abs(live.info().shared_tokens + live.info().stream_tokens + delta * n - built) * 100 > 25 * built)
        tree.append_token([5_000_000 + step * 64 + s for s in range(n)])
        delta += 1
    assert 3 <= rebuilds <= 12
    assert worst <= 0.10, worst
    if cfg == 0:
        assert worst_never > 0.3


@pytest.mark.parametrize("n_seqs,heads,root,want", [
    (4, 12, 256, 2), (4, 12, 64, 1), (2, 8, 1024, 8), (16, 32, 512, 4), (17, 32, 512, 2), (2, 32, 1024, 4),
    (16, 12, 1024, 4), (32, 12, 1024, 8), (64, 8, 1024, 4), (64, 8, 512, 4), (2, 8, 2048, 8), (2, 8, 1088, 4)])
def test_tiny_launches_cut_shared_runs_into_two_tiles(n_seqs, heads, root, want):
    """Segments of 128 shared tokens while the launch has compute units to spare, of 256 otherwise; each segment
    is attended once for every covered sequence either way."""
    rows = [(i, 64, 0, n_seqs) for i in range(root // 64)] + [(100 + s, 30, s, s + 1) for s in range(n_seqs)]
    plan = capi.build_tables(np.array(rows, np.int32), n_seqs, 64, n_heads=heads, n_cus=256)["plan"]
    items = plan["shared_items"]
    assert len(set(items[:, 4])) == want                       # ordinals of partial rows = segments
    for s in range(n_seqs):
        covering = items[(items[:, 0] <= s) & (s < items[:, 0] + items[:, 1])]
        assert sorted(covering[:, 4]) == list(range(want)) and covering[:, 3].sum() == root // 64


def test_tiny_launches_count_the_segments_that_are_cut():
    """Chunks of 32: 17 make four segments of two tiles (the nearest number), which is not more than four, though a
    fifth begins."""
    rows = [(i, 32, 0, 16) for i in range(17)] + [(100 + s, 20, s, s + 1) for s in range(16)]
    plan = capi.build_tables(np.array(rows, np.int32), 16, 32, n_heads=16, n_cus=256)["plan"]
    assert len(set(plan["shared_items"][:, 4])) == 4


def paths_of(rows, n_seqs):
    return [[r[0] for r in rows.tolist() if r[2] <= s < r[3]] for s in range(n_seqs)]


@pytest.mark.parametrize("c,shared,privates,fits", [
    (4, 8, [1, 3, 4, 5, 17], True), (4, 0, [2], True), (2, 0, [3] * 64, True), (2, 0, [3] * 65, False),
    (2, 0, [127], True), (2, 0, [127, 1], True), (2, 0, [129], False),                     # 64 chunks a path
    (2, 8, [15] * 64, True), (2, 8, [15] * 63 + [17], False),                              # 768 slots in all
])
def test_whole_paths_through_rollovers(c, shared, privates, fits):
    """What a small forward in one launch takes instead of work items: every sequence's chunks in path order, while
    sequences and chunks are few enough, and nothing from the first table on that is past one of those lines."""
    tree = capi.Tree(c, 4096)
    n = len(privates)
    for s, p in enumerate(privates):
        tree.add_seq(list(range(shared)) + [1000 * (s + 1) + t for t in range(p)])
    tree.reserve_tails()
    live = capi.HostTables(tree.get_chunks(), n, c)
    delta = 0
    for step in range(2 * c + 2):
        seqs, slots = tree.reserve_tails()
        if seqs:
            live.roll_tails(delta, seqs, slots)
            delta = 0
        want, plan = paths_of(tree.get_chunks(), n), live.plan()
        stride = max(map(len, want))
        held = n <= 64 and stride <= 64 and n * stride <= 768
        if step == 0:
            assert held == fits
        assert plan["path_stride"] == (stride if held else 0)
        assert plan["path_len"].tolist() == ([len(w) for w in want] if held else [])
        for s in range(n if held else 0):
            assert plan["paths"][s, :len(want[s])].tolist() == want[s] and not plan["paths"][s, len(want[s]):].any()
        tree.append_token([10 ** 6 + step * 100 + s for s in range(n)])
        delta += 1
