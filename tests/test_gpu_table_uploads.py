"""When device tables are brought to the device and on whose stream: tables built under stream capture, which are on
the device only once the graph has run, and those of small forwards, which whoever reads them uploads."""
import numpy as np
import pytest
import torch

from chunk_attn.capi import HostTables
from gpu_helpers import assert_close, dev, make_attention, oracle_output, to_dev

pytestmark = pytest.mark.gpu

H, C = 4, 64


def rand(rng, *shape):
    return rng.standard_normal(shape).astype(np.float16)


def cache(rng, shared, privates, general):
    attn = make_attention(H, C, sum((shared + p) // C + 3 for p in privates))
    if general:
        attn.ctx.set_plan(stream_chunks=4)    # explicit item sizes: never the direct form
    ks, vs = rand(rng, shared, H, 128), rand(rng, shared, H, 128)
    for s, p in enumerate(privates):
        k, v = np.concatenate([ks, rand(rng, p, H, 128)]), np.concatenate([vs, rand(rng, p, H, 128)])
        attn.add_seq(list(range(shared)) + [10_000 * (s + 1) + t for t in range(p)], to_dev(k), to_dev(v))
    return attn


def stream():
    return torch.cuda.current_stream().cuda_stream


# tables of one kernel argument and of several; partition 1 of the first would be the direct form's in partition 0
@pytest.mark.parametrize("privates,general", [([30, 70, 90], False), ([30, 70, 90], True), ([20 + 9 * s for s in range(70)], False)])
@pytest.mark.parametrize("timing", [0, 1, 2])
def test_eager_forwards_beside_tables_that_only_a_graph_uploads(privates, general, timing):
    rng = np.random.default_rng(len(privates))
    attn = cache(rng, 128, privates, general)
    n = len(privates)
    q = rand(rng, n, H, 128)
    qd, want = to_dev(q), oracle_output(attn, q, exact=True)
    for partition in (1, 2, 0):                        # buffers of every size are there: nothing is allocated below
        attn.forward(qd, partition)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        captured = attn.forward(qd, 1)
    attn.ctx.set_timing(timing)
    assert_close(attn.forward(qd, 1), want)            # the graph has not run yet
    for partition in (0, 2, 1, 0):
        graph.replay()
        torch.cuda.synchronize()
        assert_close(captured, want)
        assert_close(attn.forward(qd, partition), want)
    for _ in range(5):                                 # the staging buffers come round again
        attn.refresh_kernel_context(force=True)
        assert_close(attn.forward(qd), want)
    graph.replay()
    torch.cuda.synchronize()
    assert_close(captured, want)


@pytest.mark.parametrize("privates", [[30, 70, 90], [20 + 9 * s for s in range(70)]])
def test_a_captured_refresh_leaves_every_reader_its_tables(privates):
    rng = np.random.default_rng(1)
    attn = cache(rng, 128, privates, True)
    n = len(privates)
    q, k, v = rand(rng, n, H, 128), to_dev(rand(rng, n, H, 128)), to_dev(rand(rng, n, H, 128))
    qd, want = to_dev(q), oracle_output(attn, q, exact=True)
    out = torch.empty(n, H, 128, dtype=torch.float16, device=dev())
    attn.forward(qd)
    side = torch.cuda.Stream()

    def captured(call):
        attn.refresh_kernel_context(force=True)        # whatever a graph owns is replaced outside the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            attn.refresh_kernel_context(force=True)
            call()
        return graph

    noalloc = lambda: attn.ctx.attention_noalloc(qd.data_ptr(), out.data_ptr(), n, stream())   # noqa: E731
    graph = captured(noalloc)
    noalloc()                                          # eagerly, before the graph has run
    assert_close(out, want)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert_close(out, want)
    captured(lambda: None)
    attn.append_token(list(range(n)), k, v)
    q2 = rand(rng, n, H, 128)
    assert_close(attn.forward(to_dev(q2)), oracle_output(attn, q2, exact=True))
    captured(lambda: None)
    got = attn.decode_step(list(range(n)), to_dev(q2), k, v)
    assert_close(got, oracle_output(attn, q2, exact=True))


def test_readers_on_streams_that_only_know_of_the_refresh():
    """A small forward's tables are uploaded by their readers.  Two of them on streams of their own, both ordered behind
    the refresh and in no order between themselves: the second must not count on the first one's upload, which is held
    up here."""
    rng = np.random.default_rng(2)
    attn = cache(rng, 128, [30, 70, 90], False)
    other = rand(rng, 40, H, 128)
    attn.forward(to_dev(rand(rng, 3, H, 128)), 1)      # older tables in the buffer
    attn.add_seq(list(range(5000, 5040)), to_dev(other), to_dev(other))
    q, k, v = rand(rng, 4, H, 128), to_dev(rand(rng, 4, H, 128)), to_dev(rand(rng, 4, H, 128))
    qd, want = to_dev(q), oracle_output(attn, q, exact=True)
    first, second, back = (torch.cuda.Stream() for _ in range(3))
    attn.refresh_kernel_context()
    refreshed = torch.cuda.Event()
    refreshed.record()
    with torch.cuda.stream(first):
        refreshed.wait()
        torch.cuda._sleep(20_000_000)
        attn.ctx.append_kv(k.data_ptr(), v.data_ptr(), 4, stream())     # rows that nobody attends yet
    outs = []
    for side in (second, back):
        with torch.cuda.stream(side):
            refreshed.wait()
            out = torch.empty_like(qd)
            attn.ctx.attn_chunks_first(qd.data_ptr(), 4, stream())
            attn.ctx.attn_seqs_first(qd.data_ptr(), out.data_ptr(), 4, stream())
            side.synchronize()
            outs.append(out)
    assert not first.query()                           # the first reader's upload is still to come
    for out in outs:
        assert_close(out, want)
    torch.cuda.synchronize()
    attn.tree.append_token([1, 2, 3, 4])
    attn.ctx.delta_tokens = 1
    assert_close(attn.forward(qd), oracle_output(attn, q, exact=True))


def test_a_graph_brings_its_tables_whatever_was_uploaded_before():
    """An append captured behind an eager one on the same stream, replayed on another."""
    rng = np.random.default_rng(3)
    attn = cache(rng, 128, [30, 70, 90], False)
    q, k, v = rand(rng, 3, H, 128), to_dev(rand(rng, 3, H, 128)), to_dev(rand(rng, 3, H, 128))
    qd = to_dev(q)
    attn.forward(qd, 1)
    attn.refresh_kernel_context(force=True)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        attn.append_token([1, 2, 3], k, v)
        side.synchronize()
    with torch.cuda.graph(graph, stream=side):
        attn.ctx.append_kv(v.data_ptr(), k.data_ptr(), 3, stream())
    attn.tree.append_token([4, 5, 6])
    attn.ctx.delta_tokens = 2
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert_close(attn.forward(qd), oracle_output(attn, q, exact=True))


def table_bytes(attn, n):
    """Of the blob that a refresh brings to the device: its seven tables in whole 64-byte lines."""
    plan = HostTables(attn.tree.get_chunks(), n, C, stream_chunks=4, n_heads=H).plan()
    return sum(-(-plan[name].nbytes // 64) * 64 for name in ("shared_items", "stream_items", "slots", "seq_len", "part_ptr",
                                                             "tail_slot", "tail_fill"))


# tables of one to four kernel arguments of 3.5 KB and past them
@pytest.mark.parametrize("n,arguments", [(30, 1), (38, 1), (75, 2), (112, 3), (148, 4), (190, 5)])
def test_tables_of_several_kernel_arguments(n, arguments):
    """Every step another sequence's last chunk rolls over.  A device that is asked for all steps before it has run the first
    one, each with tables of its own in the same buffer, gives what one step at a time does."""
    runs = []
    for ahead in (False, True):
        rng = np.random.default_rng(n)
        attn = cache(rng, 64, [3 + 5 * s % 61 for s in range(n)], True)
        inputs = [[rand(rng, n, H, 128) for _ in range(3)] for _ in range(9)]
        on_device = [[to_dev(t) for t in step] for step in inputs]
        attn.refresh_kernel_context(force=True)        # buffers: nothing is allocated below
        torch.cuda.synchronize()
        if ahead:
            torch.cuda._sleep(60_000_000)
            slept = torch.cuda.Event()
            slept.record()
        outs = []
        for step in range(9):
            outs.append(attn.decode_step([50_000_000 + 1000 * step + s for s in range(n)], *on_device[step]))
            if not ahead:
                assert_close(outs[-1], oracle_output(attn, inputs[step][0], exact=True))
                assert -(-table_bytes(attn, n) // 3584) == arguments
            if step < 8:
                attn.refresh_kernel_context(force=True)
        if ahead and arguments <= 4:                   # (larger ones wait for a staging buffer)
            assert not slept.query()
        torch.cuda.synchronize()
        runs.append(outs)
    assert all(torch.equal(a, b) for a, b in zip(*runs))
    assert_close(attn.forward(on_device[-1][0]), oracle_output(attn, inputs[-1][0], exact=True))
