"""The direct form of small forwards (one launch, a workgroup a (sequence, head), no device tables) against the
general path and the oracle: lengths around its 64-token tiles and eight waves, every chunk size, heads and
sequences around the lines of its rule, the fused decode step with its row write, and captured launches that are
the first to read the device tables (which the direct form itself does not upload)."""
import numpy as np
import pytest
import torch

from gpu_helpers import assert_close, dev, host_state, make_attention, oracle_output, to_dev
from oracle.attention_ref import textbook_partials

pytestmark = pytest.mark.gpu


def rand(rng, *shape):
    return rng.standard_normal(shape).astype(np.float16)


def build(rng, H, c, shared, privates, general=False, kv=None):
    """kv: the rows of an earlier build, so that two caches hold the same."""
    total = sum((shared + p) // c + 3 for p in privates)
    attn = make_attention(H, c, total)
    if general:
        attn.ctx.set_plan(stream_chunks=4)    # explicit item sizes: the general path
    kv = kv or [(rand(rng, shared + max(privates), H, 128), rand(rng, shared + max(privates), H, 128)) for _ in privates]
    for s, p in enumerate(privates):
        n = shared + p
        k, v = (np.concatenate([kv[0][i][:shared], kv[s][i][shared:n]]) for i in range(2))
        attn.add_seq(list(range(shared)) + [10_000 * (s + 1) + t for t in range(p)], to_dev(k), to_dev(v))
    return attn, kv


@pytest.mark.parametrize("H,c,shared,privates", [
    (1, 64, 0, [1]), (12, 64, 256, [100, 75, 63, 1]), (5, 64, 64, [64, 65, 127, 447, 448, 449]),
    (4, 32, 96, [1, 31, 32, 33, 64, 200]), (3, 128, 128, [1, 63, 64, 65, 127, 128, 300]),
    (4, 64, 64, [7] * 64),                    # as many sequences and workgroups as it takes
    (1, 64, 0, [5] * 20 + [700]),             # the large argument block
    (32, 64, 1024, [130, 200, 10, 64, 1, 2, 3, 4]),   # long paths while half the compute units have a workgroup
    (4, 64, 704, [64] * 3), (4, 64, 704, [65] * 3),   # both sides of the line on the path's length
    (4, 64, 64, [7] * 65), (257, 64, 0, [30]),        # past the lines on sequences and workgroups
])
def test_direct_and_general_forwards_agree(H, c, shared, privates):
    rng = np.random.default_rng(len(privates) + H)
    attn, kv = build(rng, H, c, shared, privates)
    other, _ = build(rng, H, c, shared, privates, True, kv)
    q = rand(rng, len(privates), H, 128)
    got, general = attn.forward(to_dev(q)), other.forward(to_dev(q))
    # two roundings to fp16 of sums that differ by the general path's fp16 probabilities
    assert_close(got, general.float().cpu().numpy())
    assert_close(got, oracle_output(attn, q, exact=True))


@pytest.mark.parametrize("c,H,shared,privates", [(c, 4, 2 * c, [1, c - 2, c, c + 5]) for c in (32, 64, 128)] + [
    # nothing to merge: steps and forwards in different forms of one launch, up to and past four tiles
    (32, 60, 0, [1, 33, 60, 222]), (64, 60, 0, [1, 60, 130, 250]), (128, 60, 0, [1, 100, 127, 126]), (64, 8, 0, [60]),
])
def test_fused_steps_write_their_rows_and_follow_rollovers(c, H, shared, privates):
    rng = np.random.default_rng(c)
    fused, kv = build(rng, H, c, shared, privates)
    apart, _ = build(rng, H, c, shared, privates, False, kv)
    n = len(privates)
    for step in range(c + 6):
        tokens = [10 ** 6 + 100 * step + s for s in range(n)]
        q, k, v = (to_dev(rand(rng, n, H, 128)) for _ in range(3))
        out = fused.decode_step(tokens, q, k, v)
        apart.append_token(tokens, k, v)
        assert torch.equal(out, apart.forward(q))
        fills = {r[1] for r in fused.get_chunks().tolist() if r[3] - r[2] == 1}
        if step < 2 or fills & {1, c}:                 # around roll-overs: also against what takes no work list of ours
            assert_close(out, oracle_output(fused, q.cpu().numpy(), exact=True))
    rows_a, ka, va = host_state(fused)
    rows_b, kb, vb = host_state(apart)
    np.testing.assert_array_equal(rows_a, rows_b)
    for slot, n_tok in {(r[0], r[1]) for r in rows_a.tolist()}:
        np.testing.assert_array_equal(ka[slot][:, :n_tok], kb[slot][:, :n_tok])
        np.testing.assert_array_equal(va[slot][:, :n_tok], vb[slot][:, :n_tok])


def test_captured_append_before_any_upload():
    """An append recorded into a graph brings the tables along; neither eager work nor later tables may depend on
    whether the graph has run."""
    rng = np.random.default_rng(3)
    H, c, privates = 4, 64, [10, 20, 30]
    attn, kv = build(rng, H, c, 64, privates)
    q = rand(rng, 3, H, 128)
    attn.refresh_kernel_context()
    k, v = to_dev(rand(rng, 3, H, 128)), to_dev(rand(rng, 3, H, 128))
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        attn.ctx.append_kv(k.data_ptr(), v.data_ptr(), 3, torch.cuda.current_stream().cuda_stream)
    attn.tree.append_token([1, 2, 3])
    attn.ctx.delta_tokens = 1
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert_close(attn.forward(to_dev(q)), oracle_output(attn, q, exact=True))
    # eager, after the capture: the tables are uploaded for it
    attn.append_token([4, 5, 6], k, v)
    assert_close(attn.forward(to_dev(q)), oracle_output(attn, q, exact=True))
    # other tables, which a replay must leave alone: a replay writes the rows it was captured with and no more
    attn.add_seq([7] * 40, to_dev(rand(rng, 40, H, 128)), to_dev(rand(rng, 40, H, 128)))
    attn.append_token([8, 9, 10, 11], to_dev(rand(rng, 4, H, 128)), to_dev(rand(rng, 4, H, 128)))
    graph.replay()
    k4, v4 = to_dev(rand(rng, 4, H, 128)), to_dev(rand(rng, 4, H, 128))
    attn.append_token([12, 13, 14, 15], k4, v4)
    q4 = rand(rng, 4, H, 128)
    assert_close(attn.forward(to_dev(q4)), oracle_output(attn, q4, exact=True))


def test_phases_and_partitions_upload_what_they_read():
    rng = np.random.default_rng(4)
    attn, _ = build(rng, 4, 64, 128, [30, 70, 90])
    q = rand(rng, 3, 4, 128)
    want = oracle_output(attn, q, exact=True)
    qd, out = to_dev(q), torch.empty(3, 4, 128, dtype=torch.float16, device=dev())
    attn.refresh_kernel_context()
    stream = torch.cuda.current_stream().cuda_stream
    attn.ctx.attn_chunks_first(qd.data_ptr(), 3, stream)
    attn.ctx.attn_seqs_first(qd.data_ptr(), out.data_ptr(), 3, stream)
    assert_close(out, want)
    for partition in (0, 1, 0, 2, 0):
        assert_close(attn.forward(qd, partition), want)


def test_stream_hint_and_side_streams_change_no_bit():
    rng = np.random.default_rng(8)
    attn, _ = build(rng, 12, 64, 256, [100, 75, 63, 1])
    q = to_dev(rand(rng, 4, 12, 128))
    want, side = attn.forward(q), torch.cuda.Stream()
    torch.cuda.synchronize()
    for hint in (1, 2, 0):
        attn.ctx.set_stream_hint(hint)
        with torch.cuda.stream(side):
            got = attn.forward(q)
        side.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("c", [32, 64, 128])
def test_delta_tokens_past_the_room_of_last_chunks(c):
    """Set beyond what a last chunk holds, delta_tokens ends at the chunk's end, whatever the neighbours' lengths."""
    rng = np.random.default_rng(5)
    privates = [c - 4, 2 * c + 22, 3 * c, 1]
    attn, kv = build(rng, 4, c, c, privates)
    other, _ = build(rng, 4, c, c, privates, True, kv)
    for a in (attn, other):                                    # rows that nobody has written yet, the same in both
        a.refresh_kernel_context()
        for k, v, slot, n in [(*a.pool_views(), r[0], r[1]) for r in a.get_chunks().tolist()]:
            k[slot][:, n:] = torch.arange(c - n, device=dev()).half()[None, :, None] / 64
            v[slot][:, n:] = 1 - torch.arange(c - n, device=dev()).half()[None, :, None] / 64
    q = to_dev(rand(rng, 4, 4, 128))
    for delta in (0, 1, 4, 5, 11, c - 1, c, 5 * c, 1 << 20):
        attn.ctx.delta_tokens = other.ctx.delta_tokens = delta
        assert_close(attn.forward(q), other.forward(q).float().cpu().numpy())


def test_timed_forwards_run_what_they_time():
    """Mode 1: the forward as it is, here one launch; mode 2: the three phases.  The output is the same."""
    rng = np.random.default_rng(6)
    attn, _ = build(rng, 12, 64, 256, [100, 75, 63, 1])
    q = to_dev(rand(rng, 4, 12, 128))
    plain, out = attn.forward(q), torch.empty_like(q)
    for mode in (1, 0, 2):
        attn.ctx.set_timing(mode)
        for _ in range(3):
            assert torch.equal(attn.forward(q), plain)
        assert attn.ctx.read_timing()["calls"] == (3 if mode else 0)
    of_mode_2 = attn.ctx.read_partials_raw()                           # what the phases have left
    stream = torch.cuda.current_stream().cuda_stream
    attn.ctx.attn_chunks_first(q.data_ptr(), 4, stream)
    attn.ctx.attn_seqs_first(q.data_ptr(), out.data_ptr(), 4, stream)
    used = np.r_[0, 1, 4:132]
    np.testing.assert_array_equal(of_mode_2[:, :, used], attn.ctx.read_partials_raw()[:, :, used])


def test_partial_rows_are_those_of_the_last_forward():
    """A direct launch has none: none are handed out, least of all older ones."""
    rng = np.random.default_rng(7)
    attn, _ = build(rng, 3, 64, 64, [100, 75])
    q = to_dev(rand(rng, 2, 3, 128))
    stream = torch.cuda.current_stream().cuda_stream
    phases = torch.empty_like(q)
    for again in range(2):
        attn.forward(q)
        for read in (attn.ctx.read_partials_raw, attn.ctx.export_partials):
            with pytest.raises(RuntimeError, match="no partial rows"):
                read()
        attn.ctx.attn_chunks_first(q.data_ptr(), 2, stream)
        maxs, sums, attns = attn.ctx.export_partials()
        rows, kp, vp = host_state(attn)
        slot, n_tok, b, e = rows[0].tolist()
        m, l, o = textbook_partials(q.float().cpu().numpy(), slot, n_tok, b, e, kp, vp)
        np.testing.assert_allclose(maxs.reshape(m.shape), m, atol=1e-3, rtol=1e-3)      # as with explicit item sizes
        np.testing.assert_allclose(sums.reshape(l.shape), l, atol=1e-3, rtol=2e-3)
        np.testing.assert_allclose(attns.reshape(o.shape), o, atol=1e-2, rtol=1e-2)
        attn.ctx.attn_seqs_first(q.data_ptr(), phases.data_ptr(), 2, stream)
        assert np.isfinite(attn.ctx.read_partials_raw()[:, :, :2]).all()
    attn.forward(q, 1)
    assert attn.ctx.read_partials_raw().shape[1] == 3


def poison(attn, infinite):
    """NaN in every row that no token stands in; key element 0 of token t of sequence s as infinite[s, t] says."""
    kp, vp = attn.pool_views()
    c = attn.chunk_size
    for slot, n, _, _ in attn.get_chunks().tolist():
        kp[slot][:, n:], vp[slot][:, n:] = float("nan"), float("nan")
    paths = [[r[0] for r in attn.get_chunks().tolist() if r[2] <= s < r[3]] for s in range(attn.tree.n_seqs)]
    for (s, t), value in infinite.items():
        kp[paths[s][t // c]][:, t % c, 0] = value


def same(got, want):
    with np.errstate(invalid="ignore"):
        np.testing.assert_allclose(got.float().cpu().numpy(), want, atol=2e-3, rtol=1e-2, equal_nan=True)


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("c", [32, 64, 128])
def test_infinite_scores_and_stale_rows(c):
    """A key whose score is minus infinity weighs nothing, also where a tile has no other and the tile is its wave's
    first; a sequence of nothing else has no answer, nor one with a score of plus infinity.  Rows behind the last
    token are not looked at."""
    rng = np.random.default_rng(c)
    low, high = -float("inf"), float("inf")
    privates = [258, 400, 70, 700, 321, 300]
    attn, _ = build(rng, 3, c, 0, privates)
    poison(attn, {**{(0, t): low for t in (256, 257)}, **{(1, t): low for t in range(64, 192)}, **{(2, t): low for t in range(70)},
                  (3, 5): high, **{(4, t): low for t in (0, 320)}, **{(5, t): low for t in range(1, 300)}})
    q = np.abs(rand(rng, 6, 3, 128)) + np.float16(0.1)
    want = oracle_output(attn, q, exact=True)
    assert np.isnan(want[[2, 3]]).all() and np.isfinite(want[[0, 1, 4, 5]]).all()
    same(attn.forward(to_dev(q)), want)


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("c", [32, 64, 128])
def test_fused_steps_of_infinite_scores(c):
    """Steps in direct form and forwards in the general one, over paths on which both are one launch: new tokens alone
    in their tiles, with keys of minus infinity, and one that has no other token."""
    rng = np.random.default_rng(c + 1)
    privates = [64, 128, 190, 1, 250]
    fused, kv = build(rng, 30, c, 0, privates)
    apart, _ = build(rng, 30, c, 0, privates, False, kv)
    for a in (fused, apart):
        a.reserve()
        poison(a, {(3, 0): -float("inf"), **{(4, t): -float("inf") for t in range(64)}})
    for step in range(4):
        q, k, v = (np.abs(rand(rng, 5, 30, 128)) + np.float16(0.1) for _ in range(3))
        k[:4 if step < 2 else 2, :, 0] = -np.inf
        q, k, v = map(to_dev, (q, k, v))
        tokens = [10 ** 6 + 10 * step + s for s in range(5)]
        out = fused.decode_step(tokens, q, k, v)
        apart.append_token(tokens, k, v)
        np.testing.assert_array_equal(out.cpu().numpy(), apart.forward(q).cpu().numpy())
        want = oracle_output(fused, q.cpu().numpy(), exact=True)
        assert np.isnan(want[3]).all() == (step < 2) and np.isfinite(np.delete(want, 3, 0)).all()
        same(out, want)
