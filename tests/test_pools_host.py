"""Host logic of the side stream's numbered work (conef_amd._pools.side_recorded / side_wait):
which waits are issued and which are covered by an earlier one.  No GPU: streams and events are
stand-ins that note what they are asked to do."""
import torch

from conef_amd import _pools


class FakeStream:
    def __init__(self, handle):
        self.cuda_stream = handle
        self.waited_for = []

    def wait_event(self, event):
        self.waited_for.append(event)


def test_one_wait_covers_everything_recorded_before_it():
    device = torch.device("cpu")
    _pools._SIDE_ORDER.pop(device, None)
    try:
        events = ["e%d" % i for i in range(6)]
        numbers = [_pools.side_recorded(device, e) for e in events[:4]]
        assert numbers == [1, 2, 3, 4]
        main = FakeStream(11)
        # the oldest piece of work is asked for first: the wait goes to the newest event ...
        _pools.side_wait(device, main, numbers[0])
        assert main.waited_for == ["e3"]
        # ... and covers the rest of what had been recorded by then
        for n in numbers[1:]:
            _pools.side_wait(device, main, n)
        assert main.waited_for == ["e3"]
        # work recorded afterwards needs a wait of its own, again on the newest event
        later = [_pools.side_recorded(device, e) for e in events[4:]]
        _pools.side_wait(device, main, later[0])
        assert main.waited_for == ["e3", "e5"]
        _pools.side_wait(device, main, later[1])
        assert main.waited_for == ["e3", "e5"]
        # another stream has waited for nothing yet
        other = FakeStream(12)
        _pools.side_wait(device, other, numbers[1])
        assert other.waited_for == ["e5"]
        # nothing to wait for
        _pools.side_wait(device, other, None)
        assert other.waited_for == ["e5"]
    finally:
        _pools._SIDE_ORDER.pop(device, None)


def test_release_forgets_the_numbering():
    device = torch.device("cpu")
    _pools._SIDE_ORDER.pop(device, None)
    number = _pools.side_recorded(device, "e")
    _pools.release()                    # waits for the devices it knows and drops every pool
    assert device not in _pools._SIDE_ORDER
    stream = FakeStream(5)
    _pools.side_wait(device, stream, number)      # the device was idle when the pools were dropped
    assert stream.waited_for == []


def test_a_rebuilt_round_plan_still_waits_for_the_side_stream():
    """The error tensors and the Q arena of a bucket outlive its round plan, which is replaced
    whenever the bucket's buffer moves: the top-k the replaced plan left on the side stream must
    still be waited for by the next round, and so must its copy of the Q arena."""
    from types import SimpleNamespace

    from conef_amd import _psgd_engine as engine

    device = torch.device("cpu")
    _pools._SIDE_ORDER.pop(device, None)
    try:
        state = SimpleNamespace(round_cache={}, matrix_approximation_rank=2, min_compression_rate=2)
        grads = [torch.zeros(16, 32), torch.zeros(7)]
        main = FakeStream(21)
        first = engine.plan_for(state, 0, grads, ("buffer-a",), "topk", device, lambda: main)
        assert state.round_cache[0] is first and first.count == 1 and main.waited_for == []
        # the same key: the same plan, nothing to order
        assert engine.plan_for(state, 0, grads, ("buffer-a",), "topk", device, lambda: main) is first
        # the same buffer with another layout: a new plan
        assert engine.plan_for(state, 0, grads[:1], ("buffer-a",), "topk", device, lambda: main) is not first
        first = engine.plan_for(state, 0, grads, ("buffer-a",), "topk", device, lambda: main)
        # its round left a top-k and a Gram-Schmidt of the next Q factors on the side stream
        first.topk_event = "topk-done"
        first.topk_number = _pools.side_recorded(device, "topk-done")
        # the bucket's buffer moves: a new plan, which inherits the pending top-k ...
        second = engine.plan_for(state, 0, grads, ("buffer-b",), "topk", device, lambda: main)
        assert second is not first and state.round_cache[0] is second
        assert (second.topk_number, second.topk_event) == (first.topk_number, "topk-done")
        assert main.waited_for == []
        # ... and its round waits for it before it touches the error tensors, once
        engine.wait_for_side_topk(second, device, lambda: main)
        assert main.waited_for == ["topk-done"] and second.topk_number is None
        engine.wait_for_side_topk(second, device, lambda: main)
        assert main.waited_for == ["topk-done"]
        # settle() (state_dict, clean_error) still finds the event through the new plan
        assert [p.topk_event for p in state.round_cache.values()] == ["topk-done"]
        # a pending copy of the Q arena is waited for when the plan that knew of it goes
        second.q_next_number = _pools.side_recorded(device, "q-copied")
        third = engine.plan_for(state, 0, grads, ("buffer-c",), "topk", device, lambda: main)
        assert third.q_next_number is None and main.waited_for == ["topk-done", "q-copied"]
    finally:
        _pools._SIDE_ORDER.pop(device, None)


def test_a_stale_topk_table_is_told_from_a_current_one():
    from conef_amd import _psgd_engine as engine
    tensors = [torch.zeros(8), torch.zeros(9)]
    key = tuple(t.data_ptr() for t in tensors)
    table = (key, None, None, None, None, 0.4)
    assert engine.topk_table_is_stale(None, tensors, 0.4)
    assert not engine.topk_table_is_stale(table, tensors, 0.4)
    assert engine.topk_table_is_stale(table, tensors, 0.3)                         # another ratio
    assert engine.topk_table_is_stale(table, [tensors[0], torch.zeros(9)], 0.4)    # an error tensor was replaced


class FakeBuffer:
    def __init__(self):
        self.recorded_on = []

    def record_stream(self, stream):
        self.recorded_on.append(stream)


class FakeEvent:
    def record(self, stream):
        pass


def test_every_buffer_the_side_stream_works_on_is_known_to_the_allocator(monkeypatch):
    """The Gram-Schmidt of a bucket's next Q factors reads the Q arena and writes a second buffer on the
    side stream.  Both are replaced when a caller drops the P / Q memory of a bucket, and the new ones
    have to be recorded on the side stream like the first ones were."""
    from contextlib import nullcontext
    from types import SimpleNamespace

    from conef_amd import _lib, _psgd_engine as engine

    device, main, side = torch.device("cpu"), FakeStream(31), FakeStream(32)
    monkeypatch.setattr(torch.cuda, "Event", FakeEvent)
    monkeypatch.setattr(_lib, "current_stream", lambda dev: main)
    monkeypatch.setattr(_lib, "on_stream", lambda stream: nullcontext())
    monkeypatch.setattr(_pools, "side_stream", lambda dev, index, count: side)
    monkeypatch.setattr(engine, "_workspace", lambda dev, stream, nbytes: torch.zeros(8))
    lib = SimpleNamespace(conef_psgd_q_next_f32=lambda *a: 0)
    _pools._SIDE_ORDER.pop(device, None)
    try:
        state = SimpleNamespace(round_cache={}, matrix_approximation_rank=12, min_compression_rate=2)
        plan = engine._build_round(state, [torch.zeros(64, 96)], [(64, 96)], ("key",), None)
        plan.q_next_ptrs, plan.made = [None], [SimpleNamespace(value=1)]
        monkeypatch.setattr(engine.ctypes, "byref", lambda *a: None)

        def hand_over():
            engine._orthogonalise_q_aside(plan, lib, 0.0, 256, device)

        for _ in range(2):           # the second time: a caller dropped the bucket's arenas, a round took new ones
            engine._take_arenas(plan, torch.zeros(64 * 12), torch.zeros(96 * 12))
            assert plan.q_next is None and not plan.q_next_ready
            plan.q_next, plan.qs = FakeBuffer(), [FakeBuffer()]
            hand_over()
            hand_over()
            assert plan.q_next.recorded_on == [side] and plan.qs[0].recorded_on == [side]       # once is enough
        # and the round that follows waits for that work whether or not its result is used
        plan.q_next_ready = False
        engine.wait_for_side_q(plan, device, lambda: main)
        assert len(main.waited_for) == 1 and plan.q_next_number is None
    finally:
        _pools._SIDE_ORDER.pop(device, None)


def test_errors_the_side_stream_sparsifies_are_known_to_the_allocator(monkeypatch):
    """hPowerSGD's top-k works on a bucket's error tensors on the side stream or, with several hook streams,
    on the round's own.  New tensors have to be recorded on the side stream whenever they get there, also
    when a round of the other kind saw them first, and the selection state (zeroed by one stream's
    kernels for the next call) stays with one stream."""
    from contextlib import nullcontext
    from types import SimpleNamespace

    from conef_amd import _lib, _psgd_engine as engine

    class Err:
        def __init__(self, place):
            self.place, self.recorded_on, self.device = place, [], device

        def data_ptr(self):
            return self.place

        def numel(self):
            return 100

        def record_stream(self, stream):
            self.recorded_on.append(stream)

    device, main, side = torch.device("cpu"), FakeStream(51), FakeStream(52)
    launches = []
    lib = SimpleNamespace(conef_topk_batch_workspace_bytes=lambda *a: 64, conef_topk_batch_list_bytes=lambda *a: 32,
                          conef_topk_sparsify_batch_listed_f32=lambda *a: launches.append((a[-1], a[4])) or 0)
    monkeypatch.setattr(torch.cuda, "Event", FakeEvent)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "require_device_f32", lambda t, name: None)
    monkeypatch.setattr(_lib, "current_stream", lambda dev: main)
    monkeypatch.setattr(_lib, "stream_ptr", lambda t: main.cuda_stream)
    monkeypatch.setattr(_lib, "on_stream", lambda stream: nullcontext())
    monkeypatch.setattr(_pools, "side_stream", lambda dev, index, count: side)
    monkeypatch.setattr(engine, "_workspace", lambda dev, stream, nbytes, on=None: torch.zeros(8))
    _pools._SIDE_ORDER.pop(device, None)
    try:
        state = SimpleNamespace(round_cache={}, matrix_approximation_rank=1, min_compression_rate=2)
        plan = engine._build_round(state, [torch.zeros(64, 96)], [(64, 96)], ("key",), "topk")
        first, second = [Err(1000), Err(2000)], [Err(3000), Err(4000)]

        def aside(errs):
            engine._sparsify_aside(plan, errs, 0.4, device)

        aside(first)
        aside(first)
        assert [e.recorded_on for e in first] == [[side]] * 2           # once is enough
        assert launches[0] == launches[1] and launches[0][0] == side.cuda_stream
        # a caller replaced the errors and went to several hook streams for a round, then back
        plan.topk_table = engine.topk_sparsify_all(second, 0.4, plan.topk_table)
        assert [e.recorded_on for e in second] == [[]] * 2
        aside(second)
        assert [e.recorded_on for e in second] == [[side]] * 2
        # the same tensors on another stream: a selection state of that stream's own
        kept = plan.topk_table
        plan.topk_table = engine.topk_sparsify_all(second, 0.4, plan.topk_table)
        assert plan.topk_table is not kept and launches[-1][0] == main.cuda_stream and launches[-1][1] != launches[-2][1]
    finally:
        _pools._SIDE_ORDER.pop(device, None)


def _views(flat, shapes):
    out, off = [], 0
    for shape in shapes:
        n = int(torch.Size(shape).numel())
        out.append(flat[off: off + n].view(shape))
        off += n
    return out


def test_a_bucket_of_other_tensors_over_the_same_buffer_is_another_bucket():
    """Same buffer, same count, same first and last tensor, another order in between: the tables a hook
    keeps for the bucket point at other spans."""
    from types import SimpleNamespace

    from conef_amd import _bucket, _psgd_engine as engine

    flat = torch.zeros(4 * 8 + 6 * 4 + 3 + 2 * 2)
    one = _views(flat, [(4, 8), (6, 4), (3,), (2, 2)])
    other = _views(flat, [(4, 8), (3,), (6, 4), (2, 2)])
    layout = _bucket.layout(one)
    assert layout(_views(flat, [(4, 8), (6, 4), (3,), (2, 2)])) and layout(tuple(one))
    for shapes in ([(4, 8), (4, 6), (3,), (2, 2)], [(4, 8), (24,), (3,), (2, 2)], [(4, 8), (6, 4), (3,)],
                   [(4, 8), (6, 4), (3,), (2, 2), ()], [(4, 8), (6, 4), (3, 1), (2, 2)], []):
        assert not layout(_views(torch.zeros(100), shapes)), shapes
    assert not layout(other) and not layout([1, 2, 3, 4]) and not layout(None)
    assert _bucket.layout([])([]) and _bucket.layout([torch.zeros(())])([torch.ones(())])
    state = SimpleNamespace(round_cache={}, matrix_approximation_rank=1, min_compression_rate=0.1)
    main, device = FakeStream(41), torch.device("cpu")
    plan = engine.plan_for(state, 0, one, ("buffer",), None, device, lambda: main)
    assert engine.plan_for(state, 0, _views(flat, [(4, 8), (6, 4), (3,), (2, 2)]), ("buffer",), None, device, lambda: main) is plan
    assert engine.plan_for(state, 0, other, ("buffer",), None, device, lambda: main) is not plan


def test_random_block_errors_are_found_where_they_are_now():
    """A dense error tensor that a caller gave other storage (``.data =``, ``set_``), a sketch whose cells
    were replaced in the object: the step has to follow, whatever the objects' identity says."""
    from types import SimpleNamespace

    from conef_amd import RandomBlock_hook as rb, _lib

    def table(count):
        return SimpleNamespace(items=(_lib.RandBlockItem * count)(), count=count, places=None)

    state = SimpleNamespace(use_error_compression=False)
    errors = [torch.zeros(3, 4), torch.zeros(5, 2)]
    t = table(2)
    assert rb._errors_moved(t, errors)
    rb._point_at_errors(state, t, errors)
    assert not rb._errors_moved(t, errors)
    errors[1].data = torch.ones(5, 2)
    assert rb._errors_moved(t, errors)
    rb._point_at_errors(state, t, errors)
    assert not rb._errors_moved(t, errors) and t.items[1].err == errors[1].data_ptr()
    errors[0].set_(torch.ones(3, 4))
    assert rb._errors_moved(t, errors)

    state.use_error_compression = True
    plan = SimpleNamespace(in_place=True, host_ptr=16, device=torch.zeros(4), workspace_bytes=0)
    sketches = [SimpleNamespace(cs=torch.zeros(3, 4), range=4, _plan=plan, plan=lambda: plan) for _ in range(2)]
    t = table(2)
    rb._point_at_errors(state, t, sketches)
    assert not rb._errors_moved(t, sketches)
    sketches[1].cs.data = torch.ones(3, 4)
    assert rb._errors_moved(t, sketches)
    rb._point_at_errors(state, t, sketches)
    assert not rb._errors_moved(t, sketches) and t.items[1].cs_in == sketches[1].cs.data_ptr()
    sketches[0]._plan = None                     # a sketch loaded from a checkpoint: the plan may be another one
    assert rb._errors_moved(t, sketches)


def test_sketches_are_found_where_they_are_now():
    from types import SimpleNamespace

    from conef_amd import _host

    plan = object()
    sketches = [SimpleNamespace(cs=torch.zeros(3, 4), _plan=plan) for _ in range(3)]
    errs = dict(enumerate(sketches))
    cells = _host.same_sketches(sketches, [False, False, True])
    assert cells(errs.values()) and cells(sketches) and cells(tuple(sketches))
    assert not cells({}.values()) and not cells(sketches[:2]) and not cells(None)      # dropped by the caller
    twin = SimpleNamespace(cs=sketches[1].cs, _plan=plan)
    assert not cells([sketches[0], twin, sketches[2]])
    sketches[2].cs = torch.ones(3, 4)            # the one that swaps two buffers
    assert cells(sketches)
    sketches[0]._plan = None
    assert not cells(sketches)
    sketches[0]._plan = plan
    assert cells(sketches)
    sketches[1].cs.data = torch.ones(3, 4)
    assert not cells(sketches)
    sketches[1].cs = None                        # whatever is found there: the table is built anew, and says so
    assert not cells(sketches)
    del sketches[1].cs
    assert not cells(sketches)
