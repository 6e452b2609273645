"""GPU tests at the edges of single kernel paths, against the CPU oracle (bit for bit)."""

import ctypes
import threading
import time
import weakref
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch
from torch.utils import deterministic

import cabi
import cases
from nanoep_amd import Buffer, EPConfig
from nanoep_amd._native import load_extension
from oracle import nanoep_oracle as oracle
from test_gpu_buffer_api import assert_dispatch_result, assert_same_bits
from test_gpu_cabi_parity import assert_layout, run_dispatch_combine

pytestmark = pytest.mark.gpu


# The prefetch workgroups of the slot-order walk also touch their segment's list lines and weights: list
# shares that start inside a line, windows cut short by the batch's end, lists far shorter than their
# segments (most choices masked), more lines than prefetch wavefronts (short rows, 32 choices).
@pytest.mark.parametrize(
    "tokens,hidden,experts,topk,kind",
    [(257, 256, 9, 3, "dropout"), (1025, 512, 16, 5, "sparse"), (4097, 256, 40, 32, "dropout"), (65, 7168, 256, 8, "masked"),
     (2049, 2816, 3, 1, "sparse")],
)
def test_list_and_weight_lines_of_ragged_windows(device, tokens, hidden, experts, topk, kind):
    run_dispatch_combine(device, cases.routing(kind, tokens, experts, topk, seed=tokens), hidden, experts, 1, True, True, True)


# Five choices a token and more, rows of 1024 to 4096 elements and whole windows an XCD: the prefetch workgroups touch the
# list share of a segment half the walk away.  Shares that start inside a line, a last window cut short, lists far shorter
# than their segments; one choice, one element step and one window beside the rule.
@pytest.mark.parametrize(
    "tokens,hidden,experts,topk,kind",
    [(512, 1024, 9, 5, "dropout"), (511, 4096, 40, 8, "random"), (1000, 2816, 16, 6, "sparse"), (2048, 2048, 64, 32, "dropout"),
     (512, 1024, 9, 4, "dropout"), (512, 768, 9, 5, "dropout"), (511, 4352, 9, 5, "dropout"), (513, 1024, 9, 5, "dropout")],
)
def test_list_lines_of_a_segment_half_the_walk_away(device, tokens, hidden, experts, topk, kind):
    run_dispatch_combine(device, cases.routing(kind, tokens, experts, topk, seed=hidden), hidden, experts, 1, True, True, True)


# The layout's three plans (1: every workgroup counts the batch, 2: histogram rows summed by every
# workgroup, 3: histogram rows scanned by one) at the edges of its blocks, rows and wavefront chunks: batches one
# token around a block, choices whose chunks leave lanes idle, experts around a strip of 64 and beyond the
# threads of a workgroup, histogram rows of several blocks (short rows, long batches).
@pytest.mark.parametrize("launches", [1, 2, 3])
@pytest.mark.parametrize(
    "tokens,experts,topk,hidden,alignment",
    [(1, 2, 2, 256, 1), (31, 63, 5, 1024, 4), (32, 64, 8, 1024, 1), (33, 65, 10, 1024, 16), (64, 3, 1, 7168, 1), (65, 256, 8, 7168, 128),
     (127, 40, 32, 512, 1), (129, 33, 17, 2048, 2), (257, 1030, 6, 4096, 8), (513, 8, 3, 512, 3), (700, 3839, 4, 512, 1),
     (9000, 300, 7, 256, 1), (16385, 17, 8, 512, 128)],
)
def test_layout_plans_at_their_edges(device, tuning, launches, tokens, experts, topk, hidden, alignment):
    tuning("LAYOUT_LAUNCHES", launches)
    idx = cases.routing("dropout", tokens, experts, topk, seed=tokens + topk)
    for expand in (True, False):
        metadata, counts = cabi.layout(idx.to(device), experts, alignment, expand, hidden=hidden)
        assert_layout(metadata, counts, oracle.layout(idx, experts, alignment), expand, hidden)


# Batches whose assignment wavefronts take two chunks of a block each (more than 4096 wavefronts with one): the last block
# cut short inside a wavefront's first or second chunk, an odd number of chunks a block; and one token less than it takes.
@pytest.mark.parametrize(
    "tokens,experts,topk,hidden",
    [(16385, 40, 32, 2048), (8192, 40, 32, 2048), (8193, 33, 32, 512), (65570, 24, 5, 2048), (32801, 300, 9, 4096), (140001, 5, 3, 1024)],
)
def test_layout_with_two_chunks_a_wavefront(device, tokens, experts, topk, hidden):
    idx = cases.routing("dropout", tokens, experts, topk, seed=topk)
    for expand in (True, False):
        metadata, counts = cabi.layout(idx.to(device), experts, 16, expand, hidden=hidden)
        assert_layout(metadata, counts, oracle.layout(idx, experts, 16), expand, hidden)


# One bad token anywhere in the batch is found by every plan: an id in another half of its 64 bits, a
# duplicate in the token's first and last choice, in the first and last block.
@pytest.mark.parametrize("launches", [1, 2, 3])
@pytest.mark.parametrize("token", [0, 127, 128, 771])
@pytest.mark.parametrize("bad,status", [(-2, 1), (24, 1), ((1 << 32) + 3, 1), (None, 2)])
def test_every_layout_plan_reports_bad_routing(device, tuning, launches, token, bad, status):
    tuning("LAYOUT_LAUNCHES", launches)
    idx = cases.routing("random", 772, 24, 5, seed=9)
    idx[token, 4] = idx[token, 0] if bad is None else bad
    _, counts = cabi.layout(idx.to(device), 24, 1, True, raise_on_routing=False)
    assert counts[3] == status


# A layout that is told of the rows gives the same results (which rows it reads, and that they are there, test_ahead_plan.py
# shows): rows fewer than a wavefront reads, XCD shares that end inside one, as many rows as are read and one more, one launch and
# three, 2^18 pairs and a few less.
@pytest.mark.parametrize("xcds", [0, 3, 16])
@pytest.mark.parametrize(
    "tokens,hidden,topk,launches",
    [(1, 8, 2, 0), (33, 256, 5, 0), (257, 1032, 3, 2), (2048, 2048, 8, 2), (2049, 2048, 4, 3), (4100, 2816, 6, 0), (700, 7168, 8, 1),
     (1024, 2048, 2, 0), (32768, 256, 8, 0), (32767, 256, 8, 0)],
)
def test_layout_that_reads_source_rows_ahead(device, tuning, monkeypatch, tokens, hidden, topk, launches, xcds):
    tuning("XCDS", xcds)
    tuning("LAYOUT_LAUNCHES", launches)
    library = cabi.lib()
    ahead = library.nanoep_layout_ahead
    ahead.argtypes = [*library.nanoep_layout.argtypes[:-1], ctypes.c_void_p, ctypes.c_void_p]
    x = cases.payload(tokens, hidden, seed=tokens)
    rows = x.to(device)
    monkeypatch.setattr(library, "nanoep_layout", lambda *args: ahead(*args[:-1], rows.data_ptr(), args[-1]))
    idx = cases.routing("dropout", tokens, 24, topk, seed=tokens)
    for expand in (True, False):
        metadata, counts = cabi.layout(idx.to(device), 24, 16, expand, hidden=hidden)
        assert_layout(metadata, counts, oracle.layout(idx, 24, 16), expand, hidden)
    assert_same_bits(rows, x)


# A batch of one window goes without the walk's prefetch on several XCDs, with it on one: the largest such batch and one token
# more, one token, and rows that share workgroups or wavefronts, with the count on the host and on the device.
@pytest.mark.parametrize("xcds", [0, 1])
@pytest.mark.parametrize("tokens,hidden,topk,alignment", [(1, 512, 8, 4), (256, 4096, 3, 16), (257, 4096, 3, 16), (255, 256, 8, 1), (256, 1536, 6, 128)])
def test_walk_of_a_batch_of_one_window(device, tuning, tokens, hidden, topk, alignment, xcds):
    tuning("XCDS", xcds)
    run_dispatch_combine(device, cases.routing("dropout", tokens, 24, topk, seed=hidden), hidden, 24, alignment, True, True, True)


# Sixteen held tokens a wavefront of the combine: every XCD takes a run of the groups.  Fewer workgroups than XCDs, shares that
# come out even, a last share cut short and an empty one, a last group of one token, and side workgroups in front.
@pytest.mark.parametrize("xcds", [0, 1, 3, 16])
@pytest.mark.parametrize("tokens,hidden,topk", [(1, 256, 8), (16, 4096, 7), (17, 1536, 6), (129, 520, 8), (400, 2816, 8), (1009, 512, 7)])
def test_sixteen_held_tokens_in_runs_of_groups(device, tuning, tokens, hidden, topk, xcds):
    tuning("XCDS", xcds)
    idx = cases.routing("dropout", tokens, 24, topk, seed=hidden)
    lay = oracle.layout(idx, 24, 16)
    y = cases.payload(lay.expanded_capacity, hidden, seed=tokens)
    w = cases.gate_weights(lay.expanded_capacity, 1, seed=tokens).reshape(-1)
    want, want_w = oracle.combine(y, lay.recv_metadata(True), lay.dst_slots, weights=w, do_expand=True)
    metadata, counts = cabi.layout(idx.to(device), 24, 16, True, hidden=hidden)
    got, got_w = cabi.combine(y.to(device), w.to(device), None, metadata, counts, True, poison=0xA5, units=16)
    assert_same_bits(got, want)
    assert_same_bits(got_w, want_w)


# The same with nine to fifteen tokens a wavefront: a last group of fewer tokens, shares cut short and empty, side workgroups in front.
@pytest.mark.parametrize("xcds", [0, 3])
@pytest.mark.parametrize("units", [8, 9, 12, 15])
@pytest.mark.parametrize("tokens,hidden,topk", [(9, 256, 8), (121, 1536, 6), (400, 2816, 8), (1009, 520, 7)])
def test_nine_to_fifteen_held_tokens_in_runs_of_groups(device, tuning, tokens, hidden, topk, units, xcds):
    tuning("XCDS", xcds)
    idx = cases.routing("dropout", tokens, 24, topk, seed=hidden)
    lay = oracle.layout(idx, 24, 16)
    y = cases.payload(lay.expanded_capacity, hidden, seed=tokens)
    w = cases.gate_weights(lay.expanded_capacity, 1, seed=tokens).reshape(-1)
    want, want_w = oracle.combine(y, lay.recv_metadata(True), lay.dst_slots, weights=w, do_expand=True)
    metadata, counts = cabi.layout(idx.to(device), 24, 16, True, hidden=hidden)
    got, got_w = cabi.combine(y.to(device), w.to(device), None, metadata, counts, True, poison=0xA5, units=units)
    assert_same_bits(got, want)
    assert_same_bits(got_w, want_w)


def small_case(device, seed, tokens=96, hidden=512, experts=12, topk=4):
    idx = cases.routing("dropout", tokens, experts, topk, seed=seed)
    x, w = cases.payload(tokens, hidden, seed=seed), cases.gate_weights(tokens, topk, seed=seed)
    want_x, _, want_w, lay = oracle.dispatch(x, idx, experts, w, do_expand=True)
    want, _ = oracle.combine(want_x, lay.recv_metadata(True), lay.dst_slots, do_expand=True)
    return EPConfig(experts, topk, hidden, tokens), x.to(device), idx.to(device), w.to(device), want_x, want_w, want


# More asynchronous calls on their way than there are words for their completion points (64): the rest of
# them are ordered by events, and all of them behind the caller's stream, which is busy when they are made.
@pytest.mark.parametrize("calls", [1, 63, 64, 65, 150])
def test_asynchronous_calls_beyond_the_words_for_their_completion(device, calls):
    config, x, idx, w, want_x, _, want = small_case(device, 5)
    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, weights=w, do_expand=True).handle
        late_x = torch.zeros_like(x)
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
        late_x.copy_(x)
        kept = [buffer.dispatch(late_x, handle=handle, async_op=True) for _ in range(calls)]
        for received in kept:
            received.event.current_stream_wait()
        combined = buffer.combine(kept[-1].x, handle, async_op=True)
        combined.event.current_stream_wait()
        got = combined.x.clone()
        assert_same_bits(got, want, "combine")
        for received in kept[:: max(1, calls // 8)]:
            assert_same_bits(received.x, want_x, "dispatch")


# Callers on more streams than the device has hardware queues, each with a chain of asynchronous calls, made
# round-robin: every chain is ordered, whatever the streams share.
@pytest.mark.parametrize("streams", [2, 9])
def test_asynchronous_chains_on_many_streams(device, streams):
    lanes = []
    for lane in range(streams):
        config, x, idx, w, want_x, want_w, want = small_case(device, 20 + lane, tokens=40 + lane)
        lanes.append((Buffer(None, config), torch.cuda.Stream(), x, idx, w, want))
    torch.cuda.synchronize()
    results = [None] * streams
    for step in range(6):
        for lane, (buffer, stream, x, idx, w, _) in enumerate(lanes):
            with torch.cuda.stream(stream):
                received = buffer.dispatch(x if step == 0 else results[lane].x, topk_idx=idx, weights=w, do_expand=True, async_op=True)
                received.event.current_stream_wait()
                y = received.x * 1  # the caller's own work between the calls
                # (the next step dispatches what this one combined: the sums are fed back once, then the source again)
                results[lane] = buffer.combine(y, received.handle, async_op=True)
                results[lane].event.current_stream_wait()
                if step % 2:
                    results[lane].x.copy_(x)
    torch.cuda.synchronize()
    for lane, (buffer, stream, x, idx, w, want) in enumerate(lanes):
        with torch.cuda.stream(stream):
            received = buffer.dispatch(results[lane].x, topk_idx=idx, do_expand=True, async_op=True)
            received.event.current_stream_wait()
            combined = buffer.combine(received.x, received.handle, async_op=True)
            combined.event.current_stream_wait()
        torch.cuda.synchronize()
        assert_same_bits(combined.x, want, f"lane {lane}")
        buffer.close()


# Asynchronous calls of a caller that is on the communication stream itself, waited for there and from another
# stream, behind work that keeps the communication stream busy.
@pytest.mark.parametrize("consumer", ["there", "elsewhere"])
def test_asynchronous_calls_made_on_the_communication_stream(device, consumer):
    config, x, idx, w, want_x, _, want = small_case(device, 31)
    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, weights=w, do_expand=True).handle
        elsewhere = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(buffer.comm_stream):
            torch.cuda._sleep(20_000_000)
            received = buffer.dispatch(x, handle=handle, async_op=True)
            combined = buffer.combine(received.x, handle, async_op=True)
        with torch.cuda.stream(buffer.comm_stream if consumer == "there" else elsewhere):
            received.event.current_stream_wait()
            combined.event.current_stream_wait()
            got_x, got = received.x.clone(), combined.x.clone()
        torch.cuda.synchronize()
        assert_same_bits(got_x, want_x, "dispatch")
        assert_same_bits(got, want, "combine")


# A completion event that goes away unwaited keeps the call's tensors safe from the allocator: what the call
# reads is freed and its memory asked for again while the call still waits for its stream.
@pytest.mark.parametrize("explicit_event", [False, True])
def test_a_dropped_completion_event_protects_the_calls_memory(device, explicit_event):
    config, x, idx, w, want_x, want_w, _ = small_case(device, 8, tokens=200, hidden=1024)
    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, weights=w, do_expand=True).handle
        torch.cuda.synchronize()
        source = x.clone()
        ready = None
        if explicit_event:
            ready = torch.cuda.Event()
            ready.record()
        with torch.cuda.stream(buffer.comm_stream):
            torch.cuda._sleep(20_000_000)
        received = buffer.dispatch(source, handle=handle, weights=w, async_op=True, previous_event=ready)
        payload, gates = received.x, received.topk_weights
        del received, source
        poison = [torch.full_like(x, -77.0) for _ in range(4)] + [torch.full_like(want_x, -77.0, device=device) for _ in range(4)]
        torch.cuda.synchronize()
        assert_same_bits(payload, want_x, "payload")
        assert_same_bits(gates, want_w, "weights")
        del poison


def active_bytes():
    """Memory the allocator gives to nobody: in use, or freed while a stream it was told of may still use it."""
    return torch.cuda.memory_stats()["active_bytes.all.current"]


# The same for what the call writes: results, and a fresh dispatch's handle, dropped with the event while the kernels
# that write them are to run.  (A fresh dispatch returns behind its layout: its permute may have run when the memory is asked
# for again, but the allocator has been told of it.)
@pytest.mark.parametrize("call", ["replay", "fresh", "combine"])
def test_a_dropped_completion_event_protects_the_calls_results(device, call):
    tokens, hidden, experts, topk = 2048, 4096, 16, 4
    x, idx = cases.payload(tokens, hidden, seed=8).to(device), cases.routing("random", tokens, experts, topk, seed=8).to(device)
    with Buffer(None, EPConfig(experts, topk, hidden, tokens)) as buffer:
        first = buffer.dispatch(x, topk_idx=idx, do_expand=True)
        if call != "fresh":
            with torch.cuda.stream(buffer.comm_stream):
                torch.cuda._sleep(20_000_000)
        before = active_bytes()
        if call == "combine":
            shape, handle_bytes = (tokens, hidden), 0
            result = buffer.combine(first.x, first.handle, async_op=True)
        else:
            shape, handle_bytes = (tokens * topk, hidden), 0 if call == "replay" else tokens * topk * 24
            result = buffer.dispatch(x, async_op=True, **({"handle": first.handle} if call == "replay" else {"topk_idx": idx, "do_expand": True}))
        assert result.x.shape == shape
        del result
        assert active_bytes() - before >= shape[0] * hidden * 2 + handle_bytes
        mine = [torch.full(shape, -77.0, dtype=torch.bfloat16, device=device) for _ in range(3)]
        small = [torch.full((1 << 20,), 77, dtype=torch.int64, device=device) for _ in range(3)]
        torch.cuda.synchronize()
        for tensor in mine:
            assert bool((tensor == -77.0).all())
        for tensor in small:
            assert bool((tensor == 77).all())


# Early outputs that do not fit what routing filled are replaced by exact ones while the kernel that writes them may
# still be running: an asynchronous call holds them until it has been waited for, and what the caller
# allocates and fills before that stays as it was filled.  `first` makes the forecast that the second batch misses.
@pytest.mark.parametrize(
    "tokens,hidden,experts,topk,expand,alignment,first",
    [(4096, 4096, 16, 4, True, 1, None), (8192, 4096, 16, 1, False, 1, None), (2048, 4096, 64, 4, True, 128, "random")],
)
def test_replaced_early_outputs_stay_the_calls_until_it_is_waited_for(device, tokens, hidden, experts, topk, expand, alignment, first):
    x, w = cases.payload(tokens, hidden, seed=3), cases.gate_weights(tokens, topk, seed=3)
    idx = cases.routing("sparse", tokens, experts, topk, seed=3)
    x_dev, idx_dev, w_dev = x.to(device), idx.to(device), w.to(device)
    with Buffer(None, EPConfig(experts, topk, hidden, tokens)) as buffer:
        early_rows = tokens * topk if expand else tokens
        if first is not None:
            seen = buffer.dispatch(x_dev, topk_idx=cases.routing(first, tokens, experts, topk, seed=4).to(device), weights=w_dev,
                                   do_expand=expand, alignment=alignment).handle.layout.expanded_capacity
            early_rows = seen + (seen + 7) // 8
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        received = buffer.dispatch(x_dev, topk_idx=idx_dev, weights=w_dev, do_expand=expand, alignment=alignment, async_op=True)
        held = torch.cuda.memory_allocated() - before
        mine = [torch.full((early_rows, hidden), -77.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
        assert received.x.shape[0] * 5 < early_rows * 4
        early_bytes = early_rows * hidden * 2
        assert held >= early_bytes + received.x.numel() * 2
        received.event.current_stream_wait()
        assert torch.cuda.memory_allocated() - before < held + early_bytes * 2  # given back: `mine` is the two besides
        assert_dispatch_result(received, x, idx, w, experts, expand, alignment, False)
        for tensor in mine:
            assert bool((tensor == -77.0).all())


# A fresh dispatch learns of bad routing ids while its layout and the permute behind it are at work on a stream that is
# not the caller's: what they write goes back to the caller's allocator, but to nobody before they are done.
@pytest.mark.parametrize("how", [{"async_op": True}, {"num_sms": 128}], ids=["asynchronous", "budget"])
@pytest.mark.parametrize("expand", [True, False])
def test_a_call_that_fails_leaves_its_memory_to_its_kernels(device, how, expand):
    tokens, hidden, experts, topk = 4096, 4096, 16, 4
    x, idx = cases.payload(tokens, hidden, seed=6), cases.routing("random", tokens, experts, topk, seed=6)
    x_dev, idx_dev, bad_dev = x.to(device), idx.to(device), idx.to(device)
    bad_dev[tokens // 2, 1] = experts
    early_rows = tokens * topk if expand else tokens
    with Buffer(None, EPConfig(experts, topk, hidden, tokens)) as buffer:
        torch.cuda.synchronize()
        before = active_bytes()
        with pytest.raises(RuntimeError, match="out of range"):
            buffer.dispatch(x_dev, topk_idx=bad_dev, do_expand=expand, **how)
        assert active_bytes() - before >= early_rows * hidden * 2
        mine = [torch.full((early_rows, hidden), -77.0, dtype=torch.bfloat16, device=device) for _ in range(2)]
        torch.cuda.synchronize()
        for tensor in mine:
            assert bool((tensor == -77.0).all())
        del mine, tensor
        kept = torch.empty(1, device=device)  # (the allocator looks for what is done when it is asked for memory)
        assert active_bytes() - before < early_rows * hidden * 2
        received = buffer.dispatch(x_dev, topk_idx=idx_dev, do_expand=expand, **how)
        if received.event is not None:
            received.event.current_stream_wait()
        assert_dispatch_result(received, x, idx, None, experts, expand, 1, False)
        del kept


@pytest.fixture(scope="module")
def spin(device):
    """spin(milliseconds): keeps the current stream busy for about that long."""
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(100_000)
    start.record()
    torch.cuda._sleep(1_000_000)
    end.record()
    end.synchronize()
    cycles = 1_000_000 / start.elapsed_time(end)
    return lambda milliseconds: torch.cuda._sleep(int(cycles * milliseconds))


# A block of the caller's pool that another thread on the caller's stream has freed, with its kernels still to run, becomes an
# asynchronous call's result while that call is on its way: waiting for its turn behind another fresh dispatch
# (outputs made ahead of the counts), or for its counts (outputs made behind them).
@pytest.mark.parametrize("outputs", ["early", "exact"])
def test_results_come_behind_whoever_had_their_memory_last(device, spin, outputs):
    tokens, hidden, experts, topk = 2048, 4096, 16, 4
    idx = cases.routing("random" if outputs == "early" else "sparse", tokens, experts, topk, seed=14)
    x = cases.payload(tokens, hidden, seed=14)
    x_dev, idx_dev = x.to(device), idx.to(device)
    rows = tokens * topk if outputs == "early" else oracle.layout(idx, experts, 1).expanded_capacity
    mine, others = torch.cuda.Stream(), torch.cuda.Stream()

    def dispatch(stream, busy, **how):
        with torch.cuda.stream(stream):
            spin(busy)
            return buffer.dispatch(x_dev, topk_idx=idx_dev, do_expand=True, **how)

    with Buffer(None, EPConfig(experts, topk, hidden, tokens)) as buffer, ThreadPoolExecutor(2) as threads:
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        if outputs == "early":
            first = threads.submit(dispatch, others, 600)  # has the runtime's mailbox until its counts are there
            time.sleep(0.1)
        else:
            with torch.cuda.stream(buffer.comm_stream):
                spin(600)
        call = threads.submit(dispatch, mine, 0, async_op=True)
        time.sleep(0.2)
        with torch.cuda.stream(mine):
            had = torch.empty((rows, hidden), dtype=torch.bfloat16, device=device)
            where = had.data_ptr()
            spin(1000)
            had.fill_(-77.0)
            del had
        received = call.result(timeout=60)
        assert received.x.data_ptr() == where  # (else this looks at nothing)
        with torch.cuda.stream(mine):
            received.event.current_stream_wait()
        torch.cuda.synchronize()
        assert_dispatch_result(received, x, idx, None, experts, True, 1, False)
        if outputs == "early":
            assert_dispatch_result(first.result(timeout=60), x, idx, None, experts, True, 1, False)


# Waiting inside a graph's capture for a call made outside it comes to what the runtime makes of a plain event
# behind the same work, and does not depend on how the call's completion is kept.
@pytest.mark.parametrize("finished", [False, True])
def test_a_wait_inside_a_capture_is_an_events(device, finished):
    config, x, idx, w, want_x, _, _ = small_case(device, 12)

    def captures(wait):
        scratch = torch.zeros(8, device=device)
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        torch.cuda.current_stream().synchronize()
        refused = False
        with torch.cuda.stream(stream):
            graph.capture_begin(capture_error_mode="thread_local")
            try:
                scratch.add_(1)
                wait()
            except RuntimeError:
                refused = True
            try:
                graph.capture_end()
            except RuntimeError:
                refused = True
        return refused

    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, do_expand=True).handle
        if not finished:
            with torch.cuda.stream(buffer.comm_stream):
                torch.cuda._sleep(20_000_000)
        received = buffer.dispatch(x, handle=handle, async_op=True)
        plain = torch.cuda.Event()
        plain.record(buffer.comm_stream)
        if finished:
            torch.cuda.synchronize()
        assert captures(received.event.current_stream_wait) == captures(lambda: plain.wait())
        received.event.current_stream_wait()
        torch.cuda.synchronize()
        assert_same_bits(received.x, want_x, "payload")


# A synchronous call passes over a communication stream nothing was ever put on, and comes behind what the
# caller, an asynchronous call or a call with a compute-unit budget put there.
@pytest.mark.parametrize("through", ["comm_stream", "budget_stream", "async"])
def test_synchronous_calls_come_behind_the_communication_stream(device, through):
    config, x, idx, w, want_x, _, _ = small_case(device, 31)
    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, do_expand=True).handle
        late_x = torch.zeros_like(x)
        torch.cuda.synchronize()
        stream = {"comm_stream": lambda: buffer.comm_stream, "budget_stream": lambda: buffer.budget_stream(128),
                  "async": lambda: None}[through]()
        if stream is None:
            torch.cuda._sleep(20_000_000)
            late_x.copy_(x)
            first = buffer.dispatch(late_x, handle=handle, async_op=True)
            side = torch.cuda.Stream()
            with torch.cuda.stream(side):  # not ordered behind the copy but through the communication stream
                got = buffer.dispatch(late_x, handle=handle)
                got_x = got.x
            first.event.current_stream_wait()
        else:
            with torch.cuda.stream(stream):
                torch.cuda._sleep(20_000_000)
                late_x.copy_(x)
            got_x = buffer.dispatch(late_x, handle=handle).x
        torch.cuda.synchronize()
        assert_same_bits(got_x, want_x, through)


# The one-token combine for every number of rows it is made for, at rows that end inside a chunk, with all of
# bias, weights and the extra rounding, and around the batch size from which sums are held back (8192 wavefronts).
@pytest.mark.parametrize("topk", range(1, 9))
@pytest.mark.parametrize("tokens,hidden", [(3, 256), (70, 2816)])
def test_one_token_combine_for_every_row_count(device, topk, tokens, hidden):
    idx = cases.routing("sparse", tokens, 12, topk, seed=topk)
    metadata, counts = cabi.layout(idx.to(device), 12, 1, True, hidden=hidden)
    lay = oracle.layout(idx, 12, 1)
    y, bias = cases.payload(counts[1], hidden, seed=topk), cases.payload(tokens, hidden, seed=99)
    w = cases.gate_weights(counts[1], 1, seed=3).flatten()
    for multiple in (False, True):
        out, out_w = cabi.combine(y.to(device), w.to(device), bias.to(device), metadata, counts, True, multiple_reduction=multiple, poison=0xA5)
        want, want_w = oracle.combine(y, lay.recv_metadata(True), lay.dst_slots, do_expand=True, weights=w, bias=bias,
                                      multiple_reduction=multiple)
        assert_same_bits(out, want, "combine")
        assert_same_bits(out_w, want_w, "weights")


@pytest.mark.parametrize("topk", [7, 8, 9])
@pytest.mark.parametrize("tokens", [1024, 1025])
def test_combine_around_the_batch_that_holds_sums_back(device, topk, tokens):
    idx = cases.routing("dropout", tokens, 16, topk, seed=topk)
    metadata, counts = cabi.layout(idx.to(device), 16, 1, True, hidden=4096)
    lay = oracle.layout(idx, 16, 1)
    y = cases.payload(counts[1], 4096, seed=topk)
    out, _ = cabi.combine(y.to(device), None, None, metadata, counts, True, poison=0xA5)
    want, _ = oracle.combine(y, lay.recv_metadata(True), lay.dst_slots, do_expand=True)
    assert_same_bits(out, want, "combine")


# The same for the other lines of that rule: six rows of up to 2048 elements, and more than eight rows a token.
@pytest.mark.parametrize("tokens,hidden,topk", [(8191, 2048, 6), (8192, 2048, 6), (640, 4096, 16), (641, 4096, 16), (384, 4096, 17), (385, 4096, 17)])
def test_combine_around_other_batches_that_hold_sums_back(device, tokens, hidden, topk):
    idx = cases.routing("dropout", tokens, 32, topk, seed=topk)
    metadata, counts = cabi.layout(idx.to(device), 32, 1, True, hidden=hidden)
    lay = oracle.layout(idx, 32, 1)
    y, w = cases.payload(counts[1], hidden, seed=topk), cases.gate_weights(counts[1], 1, seed=3).flatten()
    out, out_w = cabi.combine(y.to(device), w.to(device), None, metadata, counts, True, poison=0xA5)
    want, want_w = oracle.combine(y, lay.recv_metadata(True), lay.dst_slots, do_expand=True, weights=w)
    assert_same_bits(out, want, "combine")
    assert_same_bits(out_w, want_w, "weights")


# Where torch is to fill uninitialized memory, a result's rows that no call writes (alignment gaps without zero padding)
# hold torch's fill value and not what their memory held before, through the native module, which accepts that mode.
@pytest.mark.parametrize("asynchronous", [False, True])
def test_deterministic_fill_reaches_the_rows_nobody_writes(device, asynchronous):
    native = load_extension()
    config, x, idx, w, _, _, _ = small_case(device, 8, tokens=200, hidden=1024)
    lay = oracle.layout(idx.cpu(), config.num_experts, 16)
    gaps = torch.ones(lay.expanded_capacity, dtype=torch.bool)
    for count, offset in zip(lay.expert_counts.tolist(), lay.expert_offsets.tolist()):
        gaps[offset : offset + count] = False
    assert bool(gaps.any())
    enabled, fill = torch.are_deterministic_algorithms_enabled(), deterministic.fill_uninitialized_memory
    warn_only = torch.is_deterministic_algorithms_warn_only_enabled()
    with Buffer(None, config) as buffer:
        torch.use_deterministic_algorithms(True)
        deterministic.fill_uninitialized_memory = True
        try:
            metadata, capacity = [], 0
            for _ in ("fresh", "cached"):
                used = [torch.full((lay.expanded_capacity, 1024), 5.0, dtype=torch.bfloat16, device=device) for _ in range(4)]
                del used
                outputs, handle, counts, event = native.dispatch(
                    buffer._runtime, x, idx, w, config.num_experts, config.num_max_tokens_per_rank, 16, metadata, capacity, False,
                    expand=True, zero_padding=False, num_sms=0, comm_stream=buffer.comm_stream.cuda_stream, async_op=asynchronous,
                )
                if event is not None:
                    event.current_stream_wait()
                assert bool(outputs[0].cpu()[gaps].isnan().all()) and not bool(outputs[0].cpu()[~gaps].isnan().any())
                assert bool(outputs[2].cpu()[gaps].isnan().all())
                metadata, capacity = (metadata or list(handle)), counts[1]
        finally:
            deterministic.fill_uninitialized_memory = fill
            torch.use_deterministic_algorithms(enabled, warn_only=warn_only)


# A synchronous call on another stream while somebody captures the communication stream: it runs, now, and the capture
# has nothing of it.
def test_synchronous_calls_beside_a_capture_of_the_communication_stream(device):
    config, x, idx, w, want_x, _, _ = small_case(device, 12)
    with Buffer(None, config) as buffer:
        handle = buffer.dispatch(x, topk_idx=idx, do_expand=True).handle
        side, stream = torch.cuda.Stream(), buffer.comm_stream
        scratch = torch.zeros(8, device=device)
        with torch.cuda.stream(side):
            buffer.dispatch(x, handle=handle)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            graph.capture_begin(capture_error_mode="relaxed")
            try:
                scratch.add_(1)
                with torch.cuda.stream(side):
                    received = buffer.dispatch(x, handle=handle).x
                    side.synchronize()
            finally:
                graph.capture_end()
        assert_same_bits(received, want_x, "dispatch")
        for _ in range(3):
            graph.replay()
        torch.cuda.synchronize()
        assert scratch.tolist() == [3.0] * 8


# What a waited-for call has read is let go of by the wait, and its end may run Python (here: a weak reference's callback)
# while another thread waits for the same call.
def test_two_threads_wait_for_a_call_whose_inputs_end_there(device):
    native = load_extension()
    config, x, idx, w, want_x, _, _ = small_case(device, 8)
    with Buffer(None, config) as buffer, ThreadPoolExecutor(2) as threads:
        handle = buffer.dispatch(x, topk_idx=idx, do_expand=True).handle
        source, ended = x.clone(), threading.Event()

        def on_end(_):
            ended.set()
            time.sleep(0.3)

        watch = weakref.ref(source, on_end)
        outputs, _, _, event = native.dispatch(
            buffer._runtime, source, idx, None, config.num_experts, config.num_max_tokens_per_rank, 1, list(handle.tensors()),
            handle.layout.expanded_capacity, False, expand=True, zero_padding=False, num_sms=0, comm_stream=buffer.comm_stream.cuda_stream,
        )
        del source
        first = threads.submit(event.current_stream_wait)
        assert ended.wait(timeout=10)
        second = threads.submit(event.current_stream_wait)
        first.result(timeout=10)
        second.result(timeout=10)
        torch.cuda.synchronize()
        assert_same_bits(outputs[0], want_x, "dispatch")
        del watch
