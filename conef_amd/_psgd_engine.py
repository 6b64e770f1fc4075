"""The per-bucket PowerSGD round shared by powerSGD_hook and hpowerSGD_hook.

Reference flow (communication/powerSGD_hook.py:338-580, hPowerSGD_hook.py:328-570):
split the bucket into matrices worth compressing and the rest; add the remembered error; P = M Q;
orthogonalise P; Q = M^T P; M = P Q^T; remember the new error.  The all-reduces that sit between
those stages in the reference are the identity at world size 1.  Here each matrix costs three
streaming passes over its memory: the error add is fused into the first product, the residual
(dense, or count-sketched) into the last.
"""
import contextlib
import ctypes
import logging
import os

import torch
import torch.distributed as dist

from . import _bucket, _host, _lib, _pools
from .compressors.CountSketch import HASH_A, HASH_B, DenseCS


def should_compress(num_rows, num_cols, matrix_approximation_rank, min_compression_rate):
    """(worth compressing?, uncompressed count, compressed count) - powerSGD_hook.py:46-70."""
    uncompressed_size = num_rows * num_cols
    compressed_size = (num_rows + num_cols) * matrix_approximation_rank
    return (compressed_size * min_compression_rate < uncompressed_size, uncompressed_size, compressed_size)


def orthogonalize(matrix, epsilon=0, workspace=None):
    """In-place Gram-Schmidt of a contiguous [rows, r] device matrix (powerSGD_hook.py:12-44)."""
    _lib.require_device_f32(matrix, "matrix")
    rows, r = matrix.shape
    lib = _lib.load()
    need = lib.conef_psgd_workspace_bytes(rows, 1, r)
    if workspace is None or workspace.numel() < need:
        workspace = _workspace(matrix.device, _lib.stream_ptr(matrix), need)
    rc = lib.conef_gram_schmidt_f32(matrix.data_ptr(), rows, r, float(epsilon), workspace.data_ptr(),
                                    workspace.numel(), _lib.stream_ptr(matrix))
    _lib.check(rc, "conef_gram_schmidt_f32")
    return workspace


def orthogonalize_all(matrices, epsilon, ws_ptr, ws_len, stream, table=None):
    """Gram-Schmidt of independent [rows, r] device matrices, side by side in as few launches as
    their shapes allow.  ``table``: what an earlier call over the same matrices returned (the host
    arrays are reused while the matrices stay where they are); returns the table."""
    count = len(matrices)
    if count == 0:
        return None
    key = tuple(m.data_ptr() for m in matrices)
    if table is None or table[0] != key:
        ptrs = (ctypes.c_void_p * count)(*key)
        rows = (ctypes.c_int64 * count)(*[m.shape[0] for m in matrices])
        ranks = (ctypes.c_int32 * count)(*[m.shape[1] for m in matrices])
        table = (key, ptrs, rows, ranks)
    _, ptrs, rows, ranks = table
    rc = _lib.load().conef_gram_schmidt_batch_f32(ptrs, rows, ranks, count, float(epsilon), ws_ptr, ws_len, stream)
    _lib.check(rc, "conef_gram_schmidt_batch_f32")
    return table


def gram_schmidt_give_ups():
    """How many Gram-Schmidt workgroups on the current device have run out their bounded wait for a
    neighbouring workgroup since the library was loaded (each leaves NaN in its rows of the factor).
    The kernels that spread one factor over several workgroups rely on those workgroups being
    resident together; with several hook streams busy that is an assumption, and this is where its
    failure shows before the NaN reaches a gradient.  Waits for the device.  With CONEF_CHECK_GS=1
    every hook call ends with this check and raises."""
    count = ctypes.c_int64(0)
    _lib.check(_lib.load().conef_gram_schmidt_give_ups(ctypes.byref(count)), "conef_gram_schmidt_give_ups")
    return count.value


# one buffer per (device, stream), grown on demand; held and released by conef_amd._pools
_workspace = _pools.workspace
_scratch_f32 = _pools.scratch_f32


def topk_sparsify(err, topk_ratio, workspace=None):
    """Keeps the max(1, int(0.5 * ratio * numel)) largest magnitudes of ``err`` in place
    (hPowerSGD_hook.py:90-97); ties on the threshold keep the lowest flat indices."""
    _lib.require_device_f32(err, "err")
    lib = _lib.load()
    numel = err.numel()
    k = max(1, int(0.5 * topk_ratio * numel))
    need = lib.conef_topk_workspace_bytes(numel)
    if workspace is None or workspace.numel() < need:
        workspace = torch.empty(need, dtype=torch.uint8, device=err.device)
    rc = lib.conef_topk_sparsify_f32(err.data_ptr(), numel, k, workspace.data_ptr(), workspace.numel(),
                                     _lib.stream_ptr(err))
    _lib.check(rc, "conef_topk_sparsify_f32")
    return workspace


class _TopkTable(tuple):
    """(tensors' places, pointers, element counts, how many stay, selection state, ratio)"""
    list_bytes = 0
    stream = None       # the raw stream the selection state was allocated and cleared on, the only one it is used on


def topk_sparsify_all(tensors, topk_ratio, table=None, side=None):
    """``topk_sparsify`` of every tensor of a list (one stream, one device) with each pass a
    single launch over all of them.  ``table`` is what an earlier call over the same tensors
    returned: the host arrays and the selection state are reused while the tensors stay where they are
    and the calls on one stream.
    ``side``: the torch Stream to launch on (the current one if None)."""
    count = len(tensors)
    if count == 0:
        return table
    lib = _lib.load()
    device = tensors[0].device
    stream = _lib.stream_ptr(tensors[0]) if side is None else side.cuda_stream
    if topk_table_is_stale(table, tensors, topk_ratio) or table.stream != stream:
        key = tuple(t.data_ptr() for t in tensors)
        for t in tensors:
            _lib.require_device_f32(t, "err")
        ptrs = (ctypes.c_void_p * count)(*key)
        numels = (ctypes.c_int64 * count)(*[t.numel() for t in tensors])
        ks = (ctypes.c_int64 * count)(*[max(1, int(0.5 * topk_ratio * t.numel())) for t in tensors])
        # zero-filled once, on the stream whose kernels rely on the zeros: the table keeps this state with
        # these tensors, and the passes clear it behind themselves (conef_topk_sparsify_batch_listed_f32)
        with contextlib.nullcontext() if side is None else _lib.on_stream(side):
            ws = torch.zeros(lib.conef_topk_batch_workspace_bytes(numels, count), dtype=torch.uint8, device=device)
        table = _TopkTable((key, ptrs, numels, ks, ws, topk_ratio))
        table.list_bytes = lib.conef_topk_batch_list_bytes(numels, count)
        table.stream = stream
    _, ptrs, numels, ks, ws, _ = table
    lists = _workspace(device, stream, table.list_bytes, side)
    rc = lib.conef_topk_sparsify_batch_listed_f32(ptrs, numels, ks, count, ws.data_ptr(), ws.numel(), lists.data_ptr(),
                                                  lists.numel(), stream)
    _lib.check(rc, "conef_topk_sparsify_batch_listed_f32")
    return table


class _RoundPlan:
    """What a bucket's round needs that does not change from step to step: which tensors are
    compressed, the table of matrices the batch entry points read, the views into the P / Q
    arenas.  Built on the first step of a bucket and reused while the bucket keeps its buffer
    and layout, so that a step costs a handful of foreign calls however many tensors it has."""
    __slots__ = ("small", "layout", "cells", "cs_static", "env_ahead", "env_topk_side", "env_small", "check_gs", "tape", "key", "shapes", "work", "passthrough", "before", "after", "total_ps", "total_qs", "arena_key", "ps",
                 "qs", "items", "count", "sketches", "fused_sketch", "fused_order", "batched_update", "residual_offsets",
                 "topk_table", "q_next", "q_next_ptrs", "q_next_ready", "q_next_made", "made", "q_next_event", "aside_recorded",
                 "topk_event", "ws_need", "handoff_event", "topk_number", "q_next_number", "is_wide", "wide", "chunks", "runs", "ef_spans")

    @property
    def q_next_fold(self):
        """Whether every run of the bucket's matrices starts its next round from what CONEF_ROUND_NEXT_FOLD asked for."""
        return bool(self.q_next_made) and all(made & 4 for made in self.q_next_made)


# flags of conef_psgd_round_ahead_f32 (include/conef_hip.h)
_ROUND_Q_READY, _ROUND_MAKE_NEXT, _ROUND_NEXT_QUADS, _ROUND_NEXT_WIDE, _ROUND_QUADS_READY = 1, 2, 4, 8, 16
_ROUND_NEXT_FOLD, _ROUND_FOLD_READY = 32, 64

BATCH_ITEMS = 24        # matrices the batch entry points take into one launch


def _chunks(count):
    """A bucket's matrices as runs of at most BATCH_ITEMS of about the same length: (first, how many)."""
    parts = -(-count // BATCH_ITEMS)
    return [(count * i // parts, count * (i + 1) // parts - count * i // parts) for i in range(parts)]


def _ef_spans(plan, base_ptr, err_ptr):
    """The stretches of a bucket that are not compressed, neighbours joined, as the host arrays
    ``conef_ef_passthrough_batch_f32`` reads: (x pointers, error pointers, element counts, how many)."""
    runs = []
    for tensor in sorted(plan.passthrough, key=lambda t: t.data_ptr()):
        at, numel = tensor.data_ptr(), tensor.numel()
        if numel == 0:
            continue
        if runs and runs[-1][0] + 4 * runs[-1][1] == at:
            runs[-1][1] += numel
        else:
            runs.append([at, numel])
    n = len(runs)
    return ((ctypes.c_void_p * n)(*[at for at, _ in runs]),
            (ctypes.c_void_p * n)(*[err_ptr + (at - base_ptr) for at, _ in runs]),
            (ctypes.c_int64 * n)(*[c for _, c in runs]), n)


def _rank_bound(rank):
    """Floats in a row of the library's own copy of a rank-r factor (ranks above 32 have none)."""
    return 1 << max(rank - 1, 0).bit_length()


def _build_round(state, grads, shapes, key, error_mode):
    plan = _RoundPlan()
    plan.key, plan.shapes = key, shapes
    plan.layout = _bucket.layout(grads)
    plan.cells = None               # the bucket's sketches as they were when the table was pointed at them
    plan.cs_static = False
    # switches read when the plan is built (a bucket's plan lives as long as its buffer does)
    plan.env_ahead = os.environ.get("CONEF_ROUND_AHEAD", "1") != "0"
    plan.env_topk_side = os.environ.get("CONEF_TOPK_SIDE", "1") != "0"
    plan.env_small = os.environ.get("CONEF_ROUND_SMALL", "1") != "0"
    plan.check_gs = _host.environment_is("CONEF_CHECK_GS", "1")      # asked every round
    plan.tape = _lib.Tape() if os.environ.get("CONEF_ROUND_TAPE", "1") != "0" else None      # the round's launches, kept (_lib.Tape)
    plan.work, plan.passthrough = [], []
    plan.before = plan.after = plan.total_ps = plan.total_qs = 0
    for tensor in grads:                                            # Step I (:394-418)
        matrix = tensor.view(tensor.shape[0], -1)
        n, m = matrix.shape
        rank = min(n, m, state.matrix_approximation_rank)
        ok, before, after = should_compress(n, m, rank, state.min_compression_rate)
        plan.before += before
        if ok:
            plan.work.append((matrix, n, m, rank))
            plan.total_ps += n * rank
            plan.total_qs += m * rank
            plan.after += after
        else:
            plan.passthrough.append(tensor)
            plan.after += before
    plan.count = len(plan.work)
    plan.items = (_lib.PsgdItem * max(plan.count, 1))()
    for cnt, (matrix, n, m, rank) in enumerate(plan.work):
        it = plan.items[cnt]
        it.x, it.n, it.m, it.r, it.w = matrix.data_ptr(), n, m, rank, 1
    plan.arena_key = None
    # a rank above 32 goes through column chunks of the factors (conef_amd/_psgd_wide.py)
    plan.is_wide = any(rank > 32 for _, _, _, rank in plan.work)
    plan.wide = None
    plan.small = None               # (mode1, mode3) -> whether the bucket's round runs as one launch (a bucket of small matrices)
    plan.sketches = []
    plan.fused_sketch = False
    plan.fused_order = None         # the order of steps it was decided for
    plan.batched_update = False
    plan.topk_table = None
    plan.topk_event = None          # the side stream's top-k of this bucket's errors, to be waited for by its next round
    plan.topk_number = None         # the side stream's running number of that top-k (None: nothing to wait for)
    plan.q_next_number = None       # likewise for the Gram-Schmidt of the next round's Q factors
    plan.ws_need = None             # bytes of workspace the batch entry points ask for (a function of the table's shapes)
    plan.handoff_event = None       # recorded on the hook's stream where the side stream may start (one event, reused)
    # Second buffer for the Q factors, orthogonalised at the end of a round for the bucket's next
    # round (conef_psgd_round_ahead_f32).  Derived data: q_memory_dict keeps what the reference
    # keeps, and the flag falls with the plan whenever the state is replaced.
    plan.q_next = plan.q_next_ptrs = None
    plan.q_next_ready = False
    plan.q_next_made = ()           # what each run's last call left there (*made of conef_psgd_round_ahead_f32)
    plan.made = None
    plan.q_next_event = None
    plan.aside_recorded = None      # the side stream (raw) that q_next and the Q arena are known to the allocator to be used on
    plan.chunks = _chunks(plan.count)
    plan.runs = [(_at(plan.items, first), part) for first, part in plan.chunks]      # the same as arguments
    plan.ef_spans = None            # dense error feedback: host arrays of the stretches that are not compressed
    plan.residual_offsets = []
    off = 0
    for _, n, m, _ in plan.work:
        plan.residual_offsets.append(off)
        off += n * m
    plan.residual_offsets.append(off)
    return plan


def _drop_q_next(plan, stream_now):
    """Gives the second buffer of the Q factors back.  Its last round may have run on another stream than the one it
    was allocated on (``hook_streams`` changed); ``stream_now()``, which the bucket's next round runs on, is ordered after that."""
    if plan.q_next is not None and stream_now is not None:
        plan.q_next.record_stream(stream_now())
    plan.q_next = None
    plan.q_next_ready = False
    plan.aside_recorded = None


def _take_arenas(plan, p_mem, q_mem, stream_now=None):
    """Points the table of matrices at the bucket's P and Q arenas.  What belonged to the arenas before -
    the second buffer of the Q factors, what the allocator was told about either - goes with them."""
    plan.ps, plan.qs, p_idx, q_idx = [], [], 0, 0
    for it, (_, n, m, rank) in zip(plan.items, plan.work):
        plan.ps.append(p_mem[p_idx: p_idx + n * rank].view(n, rank))
        plan.qs.append(q_mem[q_idx: q_idx + m * rank].view(m, rank))
        it.p, it.q = plan.ps[-1].data_ptr(), plan.qs[-1].data_ptr()
        p_idx += n * rank
        q_idx += m * rank
    plan.arena_key = (p_mem.data_ptr(), q_mem.data_ptr())
    _drop_q_next(plan, stream_now)


_side_stream = _pools.side_stream


def topk_table_is_stale(table, tensors, topk_ratio):
    """Whether ``topk_sparsify_all`` would build a new table (and allocate its workspace) for these tensors."""
    return table is None or table[0] != tuple(t.data_ptr() for t in tensors) or table[5] != topk_ratio


def plan_for(state, bucket_index, grads, key, error_mode, device, stream_now):
    """The bucket's cached round plan, rebuilt when its buffer or layout changed.  What the
    replaced plan's last round left running on the side stream works on tensors that outlive the
    plan (the error tensors in ``state.error_dict``, the Q arena): the pending top-k is handed on
    to the new plan, whose round waits for it before it touches the errors, and the stream the
    round is about to run on (``stream_now()``) is ordered after a pending copy of the Q arena
    here, since the new plan no longer knows of it."""
    plan = state.round_cache.get(bucket_index)
    if plan is None or plan.key != key or not plan.layout(grads):
        old = plan
        plan = _build_round(state, grads, [t.shape for t in grads], key, error_mode)
        if old is not None:
            plan.topk_number, plan.topk_event = old.topk_number, old.topk_event
            if old.q_next_number is not None:
                _pools.side_wait(device, stream_now(), old.q_next_number)
            _drop_q_next(old, stream_now)
        state.round_cache[bucket_index] = plan
    return plan


def wait_for_side_topk(plan, device, stream_now):
    """Orders the stream a round is about to run on after the side stream's top-k of the bucket's
    error tensors from its previous round, if one may still be running."""
    if plan.topk_number is not None:
        _pools.side_wait(device, stream_now(), plan.topk_number)
        plan.topk_number = None


def wait_for_side_q(plan, device, stream_now):
    """Orders the stream a round is about to run on after the side stream's work on the bucket's Q factors
    from its previous round: it reads the Q arena and writes ``plan.q_next``, whichever of the two the
    round goes on to use and whichever stream it runs on now."""
    if plan.q_next_number is not None:
        _pools.side_wait(device, stream_now(), plan.q_next_number)
        plan.q_next_number = None


def settle(state):
    """Orders torch's current stream after whatever the rounds of ``state`` left running on a side
    stream that touches the state's own tensors (the top-k of the error tensors): to be called
    before those tensors are read or written from outside the hooks."""
    for plan in getattr(state, "round_cache", {}).values():
        event = getattr(plan, "topk_event", None)
        if event is not None:
            torch.cuda.current_stream().wait_event(event)


def run_round(state, bucket, error_mode):
    """One hook call.  error_mode: None | 'ef' (dense, whole bucket) | 'conef' (count sketch per
    matrix) | 'conef_v2' (count sketch over the [m,n] re-view of each matrix's memory,
    powerSGD_hook.py:918-920,1074-1076) | 'topk' (dense per matrix, magnitude-sparsified).

    With ``state.hook_streams`` = N > 1 the buckets of a step are dealt out over N streams: bucket
    i with i % N == 0 stays on the stream the hook was called on, the others go to one of N - 1 side
    streams.  A side stream first waits for the hook's stream (the gradients are ready there), and
    the returned Future carries the side stream's completion event, which is what DDP (or any caller
    of ``wait()``) orders its own stream after.  (Handing a bucket to another stream costs the host
    about 30 us, more than issuing its four launches: every N-th bucket is spared that.)"""
    input_tensor = _bucket.buffer(bucket)
    streams = streams_for(state, input_tensor)
    if streams <= 1 or not input_tensor.is_cuda or state.iter < state.start_powerSGD_iter:
        return _run_round(state, bucket, input_tensor, error_mode, 1)
    device = input_tensor.device
    index = _bucket.index(bucket)
    lane = index % streams
    if lane == 0:
        return _run_round(state, bucket, input_tensor, error_mode, streams)
    side = _side_stream(device, lane - 1, streams - 1)
    # the side stream starts where the hook's stream is now (one event per side stream, recorded again
    # for every bucket: a wait takes the event as it is when the wait is enqueued)
    event = _pools.side_event(device, lane - 1, streams - 1)
    event.record(_lib.current_stream(device))
    side.wait_event(event)
    input_tensor.record_stream(side)
    with _lib.on_stream(side):
        return _run_round(state, bucket, input_tensor, error_mode, streams)


AUTO_STREAMS_MIN_NUMEL = 1 << 20


def streams_for(state, input_tensor):
    """Streams the rounds of this state's buckets are dealt out over (the hook's own included).
    ``state.hook_streams`` 0 leaves it to the bucket's size: buckets of a million elements or more
    alternate between the hook's stream and a side stream (a bucket's launches that are mostly
    latency then overlap the neighbouring bucket's streaming passes), a smaller one stays on the
    hook's stream, where handing it over would cost more than it brings."""
    streams = int(getattr(state, "hook_streams", 1) or 0)
    if streams == 0:
        streams = 2 if input_tensor.numel() >= AUTO_STREAMS_MIN_NUMEL else 1
    return streams


def _run_round(state, bucket, input_tensor, error_mode, streams):
    group, world_size = _bucket.group_and_size(state.process_group)

    if state.iter < state.start_powerSGD_iter:
        state.maybe_increase_iter(bucket)
        return _bucket.allreduce_fut(group, input_tensor, world_size)

    if world_size != 1:
        raise NotImplementedError(
            "the MI355X PowerSGD hooks run the whole round on one GPU; with %d ranks the P and Q "
            "all-reduces between the passes are not wired up" % world_size)

    _lib.require_device_f32(input_tensor, "bucket buffer")
    lib = _lib.load()
    stream = _lib.stream_ptr(input_tensor)
    device, dtype = input_tensor.device, input_tensor.dtype
    bucket_index = _bucket.index(bucket)
    total_length = input_tensor.shape[0]
    base_ptr = input_tensor.data_ptr()

    dense_err = None
    if error_mode == "ef":
        if bucket_index not in state.error_dict:
            logging.info("A zero tensor of length {} that represents local error is created.".format(total_length))
            state.error_dict[bucket_index] = torch.zeros(total_length, device=device, dtype=dtype)
        dense_err = state.error_dict[bucket_index]
    elif error_mode in ("conef", "conef_v2", "topk"):
        state.error_dict.setdefault(bucket_index, {})
    errs = state.error_dict.get(bucket_index)

    grads = _bucket.gradients(bucket)
    key = (base_ptr, total_length, error_mode, state.matrix_approximation_rank, state.min_compression_rate,
           getattr(state, "sketch_size", None), dense_err.data_ptr() if dense_err is not None else 0)
    plan = state.round_cache.get(bucket_index)
    if plan is None or plan.key != key or not plan.layout(grads):
        plan = plan_for(state, bucket_index, grads, key, error_mode, device, lambda: _lib.current_stream(device))
    work, items, count = plan.work, plan.items, plan.count
    state.total_numel_before_compression += plan.before
    state.total_numel_after_compression += plan.after

    # Step III: P and Q arenas, reused across iterations under warm start (:434-471)
    need_randomize_qs = (not state.warm_start) or bucket_index not in state.p_memory_dict
    if need_randomize_qs:
        if state.warm_start:
            logging.info("Allocating contiguous memory of length {} for Ps, and of length {} for Qs, "
                         "respectively.".format(plan.total_ps, plan.total_qs))
        state.p_memory_dict[bucket_index] = torch.empty(plan.total_ps, device=device, dtype=dtype)
        state.q_memory_dict[bucket_index] = torch.empty(plan.total_qs, device=device, dtype=dtype)
    p_mem, q_mem = state.p_memory_dict[bucket_index], state.q_memory_dict[bucket_index]
    if plan.arena_key != (p_mem.data_ptr(), q_mem.data_ptr()):
        _take_arenas(plan, p_mem, q_mem, lambda: _lib.current_stream(device))
        if plan.is_wide and plan.wide is None:
            from ._psgd_wide import WideRound
            plan.wide = WideRound(work, plan.ps, plan.qs, device)
    if need_randomize_qs:
        plan.q_next_ready = False
    qs = plan.qs

    # error memory of every matrix in the table (created on first use; pointers that can move
    # between steps are refreshed)
    alpha = 1 - state.beta if error_mode in ("conef", "conef_v2") else 0.0
    if error_mode == "ef":
        if items[0].err is None and count:
            for cnt, (matrix, n, m, rank) in enumerate(work):
                items[cnt].err = dense_err.data_ptr() + (matrix.data_ptr() - base_ptr)
    elif error_mode == "topk":
        for cnt, (matrix, n, m, rank) in enumerate(work):
            if cnt not in errs:
                errs[cnt] = torch.zeros_like(matrix)
                if plan.tape is not None:
                    plan.tape.signature = None
                plan.topk_table = None       # perhaps at the address of a dropped one, and yet another allocation
            items[cnt].err = errs[cnt].data_ptr()
    elif error_mode == "conef":
        # (the bucket's sketches, their plans, and the cells of those that are updated in place)
        if plan.cells is None or not plan.cells(errs.values()):
            plan.sketches = []
            for cnt, (matrix, n, m, rank) in enumerate(work):
                if cnt not in errs:
                    errs[cnt] = DenseCS(n, m, state.sketch_size, device=device)
                cs = errs[cnt]
                sk_plan = cs.plan()
                it = items[cnt]
                it.w = cs.range
                it.plan_host, it.plan_dev = (sk_plan.host_ptr, sk_plan.device.data_ptr()) if sk_plan is not None else (None, None)
                plan.sketches.append((cs, sk_plan))
            plan.batched_update = all(p is not None and p.batchable for _, p in plan.sketches)
            plan.small = None
            plan.ws_need = None
            _drop_q_next(plan, lambda: _lib.current_stream(device))      # sized for the sketches, and holds sums over their buckets
            # sketches on row lists are updated in place.  The others swap two buffers, so their pointers
            # are refreshed every step.
            plan.cs_static = all(p is not None and p.in_place for _, p in plan.sketches)
            moves = [p is None or not p.in_place for _, p in plan.sketches]
            plan.cells = _host.same_sketches(errs.values(), moves + [True] * (len(errs) - count))
            for cnt, (cs, _) in enumerate(plan.sketches):
                items[cnt].cs = cs.cs.data_ptr()
            plan.fused_order = None
        if not plan.cs_static:
            for cnt, (cs, _) in enumerate(plan.sketches):
                items[cnt].cs = cs.cs.data_ptr()
        # above rank 8 also a matter of the order of steps, which may be switched from step to step
        order = lib.conef_psgd_round_in_order() if state.matrix_approximation_rank > 8 else 0
        if plan.fused_order != order:
            plan.fused_order = order
            plan.fused_sketch = plan.batched_update and (state.matrix_approximation_rank <= 8 or not plan.is_wide and all(
                lib.conef_psgd_round_wide_sketch_fits(run, part, HASH_A, HASH_B) for run, part in plan.runs))
    elif error_mode == "conef_v2":
        for cnt, (matrix, n, m, rank) in enumerate(work):
            if cnt not in errs:
                errs[cnt] = DenseCS(m, n, state.sketch_size, device=device)

    # the errors this round adds to may still be being sparsified on the side stream, and the Q factors
    # it writes may still be being read there
    if plan.topk_number is not None:
        wait_for_side_topk(plan, device, lambda: _lib.current_stream(device))
    if plan.q_next_number is not None:
        wait_for_side_q(plan, device, lambda: _lib.current_stream(device))
    eps = float(state.orthogonalization_epsilon)
    if plan.ws_need is None:
        plan.ws_need = plan.wide.ws_need if plan.is_wide else max(
            [lib.conef_psgd_batch_workspace_bytes(run, part) for run, part in plan.runs] + [256])
    ws = _workspace(device, stream, plan.ws_need)
    ws_ptr, ws_len = ws.data_ptr(), ws.numel()
    if need_randomize_qs:
        # same seeded CPU draws as the reference so every replica starts from the same Q (:479-494)
        with torch.random.fork_rng(devices=[]):
            torch.manual_seed(state.rng.randint(1_000_000_000))
            host_q = [torch.randn(*q.shape, device="cpu", dtype=dtype) for q in qs]
        for q, hq in zip(qs, host_q):
            q.copy_(hq)
    if error_mode == "conef_v2":
        # the sketch sees the same memory as m rows of n columns, so its rows are not the matrix
        # rows: query as a pass of its own (P = M Q then runs without a fused error add)
        for cnt, (matrix, n, m, rank) in enumerate(work):
            errs[cnt].query(matrix.view(m, n), alpha)
    if error_mode == "ef" and plan.ef_spans is None:
        plan.ef_spans = _ef_spans(plan, base_ptr, dense_err.data_ptr())

    # The round itself, one foreign call: orthogonalise all Q side by side; pass 1, the error add
    # fused into P = M Q; orthogonalise all P; pass 2, Q = M^T P; pass 3, M = P Q^T with the
    # residual fused.
    mode1 = {"ef": 1, "topk": 1, "conef": 2}.get(error_mode, 0)
    residual = None
    if error_mode in ("ef", "topk"):
        mode3 = 1
    elif error_mode == "conef" and plan.fused_sketch:
        mode3 = 2
    elif error_mode in ("conef", "conef_v2"):
        # The residual goes out dense and the sketches are updated from it afterwards: buckets that
        # conef_psgd_round_wide_sketch_fits does not take above rank 8, sketches whose plan is not a row
        # list, and the re-viewed sketches of C2CS_hook_v2.
        residual = _scratch_f32(device, stream, max(plan.residual_offsets[-1], 1))
        for cnt in range(count):
            items[cnt].err = residual.data_ptr() + 4 * plan.residual_offsets[cnt]
        # every sketch of the bucket from its matrix's residual in one more launch, when the plans allow
        mode3 = 3 if error_mode == "conef" and plan.batched_update else 1
    else:
        mode3 = 0
    beta3 = float(state.beta) if mode3 in (2, 3) else 0.0
    topk_aside = error_mode == "topk" and count and streams <= 1 and plan.env_ahead and plan.env_topk_side

    # A step like the last one - the same tables, scalars and buffers - makes the launches the last one made
    # (_lib.Tape; the tables are compared natively).  What a round starts on other streams is not kept.
    tape = plan.tape
    if tape is not None and (need_randomize_qs or plan.is_wide or not count or error_mode == "conef_v2" or not state.warm_start
                             or mode1 == 2 and not plan.cs_static
                             or residual is not None and (mode3 != 3 or streams <= 1)
                             or state.matrix_approximation_rank > 8 and streams <= 1):
        tape = None
    if tape is not None:
        signature = (plan.q_next_ready, plan.q_next_made, mode1, mode3, alpha, beta3, eps, ws_ptr, ws_len,
                     stream, topk_aside, getattr(state, "topk_ratio", None) if error_mode == "topk" else None)
        if signature == tape.signature:
            rc = lib.conef_tape_replay(tape.handle, items, count, stream)
            if rc == 0:
                if topk_aside:
                    _sparsify_aside(plan, [errs[cnt] for cnt in range(count)], state.topk_ratio, device)
                return _end_round(state, plan, bucket, bucket_index, input_tensor)
            if rc != _lib.TAPE_STALE:
                _lib.check(rc, "conef_tape_replay")
    if plan.tape is not None:
        plan.tape.signature = None       # a round that makes its launches anew may replace what the kept ones point to
    if tape is not None and signature != tape.seen:
        tape.seen, tape.refused, tape = signature, None, None        # kept from the second such round on: a single one costs nothing more
    if tape is not None and signature != tape.refused and tape.record(lib):
        done = False
        try:
            _issue_round(state, plan, lib, errs, error_mode, mode1, mode3, alpha, beta3, eps, ws_ptr, ws_len, stream, streams, residual,
                         topk_aside, device, dtype)
            # (a round that leaves the second buffer in another state than it found it in is not the next one's;
            # nor is one whose top-k lists lie elsewhere than in this workspace)
            done = (signature[:2] == (plan.q_next_ready, plan.q_next_made)
                    and (error_mode != "topk" or topk_aside or plan.topk_table.list_bytes <= ws_len))
        finally:
            lib.conef_tape_stop(tape.handle, items, count, done)
        if done and lib.conef_tape_kept(tape.handle):
            tape.signature = signature
        else:
            tape.refused = signature
    else:
        _issue_round(state, plan, lib, errs, error_mode, mode1, mode3, alpha, beta3, eps, ws_ptr, ws_len, stream, streams, residual,
                     topk_aside, device, dtype)
    if topk_aside:
        # The sparsification only touches the error tensors, which nobody reads before this bucket's
        # next round: it runs on a side stream while this stream goes on with the next bucket
        # (streaming passes next to launches that are mostly latency).  Same kernels, same values.
        _sparsify_aside(plan, [errs[cnt] for cnt in range(count)], state.topk_ratio, device)
    return _end_round(state, plan, bucket, bucket_index, input_tensor)


def _end_round(state, plan, bucket, bucket_index, input_tensor):
    if not state.warm_start:
        state.p_memory_dict.clear()
        state.q_memory_dict.clear()

    if plan.check_gs() and gram_schmidt_give_ups():
        raise RuntimeError("a Gram-Schmidt workgroup gave up waiting for its neighbours: the factors of bucket %d hold NaN"
                           % bucket_index)
    state.maybe_increase_iter(bucket)
    return _bucket.completed_future(input_tensor)


def _issue_round(state, plan, lib, errs, error_mode, mode1, mode3, alpha, beta3, eps, ws_ptr, ws_len, stream, streams, residual,
                 topk_aside, device, dtype):
    """The launches of a round."""
    work, items, count = plan.work, plan.items, plan.count
    if error_mode == "ef" and plan.ef_spans[3]:
        # tensors that are not compressed: g += e, and their new error is exactly zero (:361,:558)
        rc = lib.conef_ef_passthrough_batch_f32(*plan.ef_spans, stream)
        _lib.check(rc, "conef_ef_passthrough_batch_f32")
    if plan.is_wide:
        # A rank above 32: the error is added in passes of its own, the round runs on column chunks of
        # the factors, and the residual leaves the round dense (a sketch is updated from it below).
        plan.small = ((mode1, mode3), False)
        plan.q_next_ready = False
        if mode3 == 3:
            mode3 = 1
        for cnt, (matrix, n, m, rank) in enumerate(work):
            if mode1 == 1:
                _lib.check(lib.conef_ef_passthrough_f32(matrix.data_ptr(), items[cnt].err, n * m, stream), "conef_ef_passthrough_f32")
            elif mode1 == 2:
                errs[cnt].query(matrix, alpha)
        dest = [items[cnt].err if mode3 == 1 else None for cnt in range(count)]
        plan.wide.run(lib, plan.ps, plan.qs, dest, eps, ws_ptr, ws_len, stream)
    elif plan.small is None or plan.small[0] != (mode1, mode3):
        # a bucket of small matrices (every one fits a workgroup's LDS with its factors): the whole round in one launch
        fits = bool(count and mode3 in (0, 1, 2) and plan.env_small
                    and all(lib.conef_psgd_round_small_fits(run, part, mode1, mode3, HASH_A, HASH_B)
                            for run, part in plan.runs))
        plan.small = ((mode1, mode3), fits)
    if plan.is_wide:
        pass
    elif plan.small[1]:
        plan.q_next_ready = False
        for run, part in plan.runs:
            rc = lib.conef_psgd_round_small_f32(run, part, mode1, mode3, float(alpha), beta3, eps, HASH_A, HASH_B,
                                                ws_ptr, ws_len, stream)
            _lib.check(rc, "conef_psgd_round_small_f32")
    elif count and state.warm_start and plan.env_ahead and (state.matrix_approximation_rank > 8 or mode3 in (0, 1, 2)):
        # The bucket's next round starts by orthogonalising the Q factors this round leaves
        # (powerSGD_hook.py:496-497): a few workgroups and an idle machine.  It is done at the end of
        # this round instead, into a second buffer: by workgroups of the last launch at ranks up to 8 and, with
        # a sketched error, at ranks 16 and 32, by short launches of their own else (CONEF_ROUND_AHEAD=0 keeps the
        # reference's order, for comparisons).  Where the buckets do not run side by side (one stream), the
        # launches above rank 8 go to a side stream, which the bucket's next round waits for, and overlap the
        # next bucket.
        if plan.q_next is None:
            # row-major factors first, then the same in the order the kernels of ranks up to 8 load them, and behind
            # that what a round with a sketched error keeps (CONEF_ROUND_NEXT_FOLD)
            by_rows = [m * _rank_bound(rank) for _, _, m, rank in work]
            by_quads = [(-(-m // 4) * 4 + (items[cnt].w + _rank_bound(rank) + 1 if mode1 == 2 else 0)) * _rank_bound(rank)
                        for cnt, (_, _, m, rank) in enumerate(work)]
            plan.q_next = torch.empty(sum(by_rows) + sum(by_quads), device=device, dtype=dtype)
            at = [plan.q_next.data_ptr()]
            for numel in by_rows + by_quads:
                at.append(at[-1] + 4 * numel)
            plan.q_next_ptrs = [(ctypes.c_void_p * (2 * part))(*at[first: first + part], *at[count + first: count + first + part])
                                for first, part in plan.chunks]
            plan.made = [ctypes.c_int32(0) for _ in plan.chunks]
            plan.q_next_ready = False
        aside = state.matrix_approximation_rank > 8 and streams <= 1
        flags = _ROUND_NEXT_QUADS | _ROUND_NEXT_WIDE | (_ROUND_NEXT_FOLD if mode1 == 2 else 0) | (0 if aside else _ROUND_MAKE_NEXT)
        # what lies there by quads and by buckets is each run's own matter
        ready = [_ROUND_Q_READY | (_ROUND_QUADS_READY if was & 2 else 0) | (_ROUND_FOLD_READY if was & 4 else 0)
                 for was in plan.q_next_made] if plan.q_next_ready else [0] * len(plan.chunks)
        for (run, part), q_next, made, was in zip(plan.runs, plan.q_next_ptrs, plan.made, ready):
            rc = lib.conef_psgd_round_ahead_f32(run, part, mode1, mode3, float(alpha), beta3, eps, HASH_A, HASH_B,
                                                q_next, flags | was, ctypes.byref(made), ws_ptr, ws_len, stream)
            _lib.check(rc, "conef_psgd_round_ahead_f32")
        plan.q_next_made = tuple(made.value for made in plan.made)
        plan.q_next_ready = all(made & 1 for made in plan.q_next_made)
        if aside:
            _orthogonalise_q_aside(plan, lib, eps, ws_len, device)
    else:
        plan.q_next_ready = False
        for run, part in plan.runs:
            rc = lib.conef_psgd_round_f32(run, part, mode1, mode3, float(alpha), beta3, eps, HASH_A, HASH_B,
                                          ws_ptr, ws_len, stream)
            _lib.check(rc, "conef_psgd_round_f32")
    if error_mode == "topk":
        if not topk_aside:
            plan.topk_table = topk_sparsify_all([errs[cnt] for cnt in range(count)], state.topk_ratio, plan.topk_table)
    elif residual is not None and mode3 != 3:
        for cnt, (matrix, n, m, rank) in enumerate(work):
            res = residual[plan.residual_offsets[cnt]: plan.residual_offsets[cnt + 1]]
            errs[cnt].update(res.view(n, m) if error_mode == "conef" else res.view(m, n), state.beta)


def _at(array, index):
    """The ctypes array from entry ``index`` on, as an argument."""
    return ctypes.byref(array, index * ctypes.sizeof(array._type_))


def _sparsify_aside(plan, tensors, topk_ratio, device):
    """The top-k of a bucket's error tensors on the side stream, which the bucket's next round waits for."""
    if plan.handoff_event is None:
        plan.handoff_event = torch.cuda.Event()
    plan.handoff_event.record(_lib.current_stream(device))
    side = _pools.side_stream(device, 0, 1)
    side.wait_event(plan.handoff_event)
    table = topk_sparsify_all(tensors, topk_ratio, plan.topk_table, side)
    if table is not plan.topk_table:
        # a new table (an error tensor was replaced, another ratio, a round on another stream before): memory
        # the side stream works on must not go back to the allocator under it
        plan.topk_table = table
        for t in tensors:
            t.record_stream(side)
    if plan.topk_event is None:
        plan.topk_event = torch.cuda.Event()
    plan.topk_event.record(side)
    plan.topk_number = _pools.side_recorded(device, plan.topk_event)


def _orthogonalise_q_aside(plan, lib, eps, ws_len, device):
    """The new Q factors of a bucket orthogonalised for its next round on the side stream."""
    if plan.handoff_event is None:
        plan.handoff_event = torch.cuda.Event()
    plan.handoff_event.record(_lib.current_stream(device))
    side = _pools.side_stream(device, 0, 1)
    side.wait_event(plan.handoff_event)
    if plan.q_next_event is None:
        plan.q_next_event = torch.cuda.Event()
    if plan.aside_recorded != side.cuda_stream:
        # memory the side stream works on must not go back to the allocator under it: the second buffer it
        # writes and the arena it reads, each time either is a new one (all of plan.qs is one allocation)
        plan.q_next.record_stream(side)
        plan.qs[0].record_stream(side)
        plan.aside_recorded = side.cuda_stream
    with _lib.on_stream(side):
        ws = _workspace(device, side.cuda_stream, max(ws_len, 256))
    for (run, part), q_next, made in zip(plan.runs, plan.q_next_ptrs, plan.made):
        rc = lib.conef_psgd_q_next_f32(run, part, eps, q_next, ctypes.byref(made),
                                       ws.data_ptr(), ws.numel(), side.cuda_stream)
        _lib.check(rc, "conef_psgd_q_next_f32")
    plan.q_next_event.record(side)
    plan.q_next_number = _pools.side_recorded(device, plan.q_next_event)
    plan.q_next_made = tuple(made.value for made in plan.made)
    plan.q_next_ready = all(plan.q_next_made)


def run_batched_round(state, bucket):
    """batched_powerSGD_hook (powerSGD_hook.py:583-787): the whole flat bucket, zero-padded to a
    square [s,s] with s = ceil(sqrt(length)), is one matrix; dense error feedback over the padded
    length; P and Q are [s, matrix_approximation_rank]."""
    import math

    group, world_size = _bucket.group_and_size(state.process_group)
    input_tensor = _bucket.buffer(bucket)
    if state.iter < state.start_powerSGD_iter:
        state.maybe_increase_iter(bucket)
        return _bucket.allreduce_fut(group, input_tensor, world_size)
    if world_size != 1:
        raise NotImplementedError(
            "the MI355X PowerSGD hooks run the whole round on one GPU; with %d ranks the P and Q "
            "all-reduces between the passes are not wired up" % world_size)
    _lib.require_device_f32(input_tensor, "bucket buffer")
    lib = _lib.load()
    stream = _lib.stream_ptr(input_tensor)
    device, dtype = input_tensor.device, input_tensor.dtype
    bucket_index = _bucket.index(bucket)
    total_length = input_tensor.shape[0]
    side = math.isqrt(total_length)
    if side * side < total_length:
        side += 1
    rank = state.matrix_approximation_rank
    state.total_numel_before_compression += total_length
    state.total_numel_after_compression += side * rank * 2
    padded = side * side
    if rank > side:
        raise ValueError("matrix_approximation_rank %d does not fit a %d x %d matrix" % (rank, side, side))

    # the bucket buffer cannot grow in place, so a padded bucket is worked on in a square buffer
    if padded == total_length:
        square = input_tensor
    else:
        square = state.batched_square_dict.get(bucket_index)
        if square is None or square.numel() != padded:
            square = torch.empty(padded, device=device, dtype=dtype)
            state.batched_square_dict[bucket_index] = square
        square[:total_length].copy_(input_tensor)
        square[total_length:].zero_()

    err = None
    if state.use_error_feedback:
        if bucket_index not in state.error_dict:
            logging.info("A zero tensor of length {} that represents local error is created.".format(padded))
            state.error_dict[bucket_index] = torch.zeros(padded, device=device, dtype=dtype)
        err = state.error_dict[bucket_index]

    if not state.warm_start or bucket_index not in state.p_memory_dict:
        if state.warm_start:
            logging.info("Initializing low-rank tensors P and Q, each of which has a shape of {} x {}.".format(
                side, rank))
        state.p_memory_dict[bucket_index] = torch.empty(side, rank, device=device, dtype=dtype)
        with torch.random.fork_rng(devices=[]):
            torch.manual_seed(state.rng.randint(1_000_000_000))
            host_q = torch.randn(side, rank, device="cpu", dtype=dtype)
        state.q_memory_dict[bucket_index] = host_q.to(device)
    p, q = state.p_memory_dict[bucket_index], state.q_memory_dict[bucket_index]

    eps = float(state.orthogonalization_epsilon)
    if rank > 32:
        # column chunks of the factors (conef_amd/_psgd_wide.py), built once per bucket and square buffer
        from ._psgd_wide import WideRound
        wide = state.round_cache.get(bucket_index)
        if wide is None or wide[0] != (square.data_ptr(), side, rank):
            wide = ((square.data_ptr(), side, rank), WideRound([(square.view(side, side), side, side, rank)], [p], [q], device))
            state.round_cache[bucket_index] = wide
        ws = _workspace(device, stream, wide[1].ws_need)
        if err is not None:
            _lib.check(lib.conef_ef_passthrough_f32(square.data_ptr(), err.data_ptr(), padded, stream), "conef_ef_passthrough_f32")
        wide[1].run(lib, [p], [q], [err.data_ptr() if err is not None else None], eps, ws.data_ptr(), ws.numel(), stream)
        if square is not input_tensor:
            input_tensor.copy_(square[:total_length])
        if not state.warm_start:
            state.p_memory_dict.clear()
            state.q_memory_dict.clear()
        state.maybe_increase_iter(bucket)
        return _bucket.completed_future(input_tensor)
    ws = _workspace(device, stream, lib.conef_psgd_workspace_bytes(side, side, rank))
    ws_ptr, ws_len = ws.data_ptr(), ws.numel()
    _lib.check(lib.conef_gram_schmidt_f32(q.data_ptr(), side, rank, eps, ws_ptr, ws_len, stream),
               "conef_gram_schmidt_f32")
    if err is not None:
        rc = lib.conef_psgd_mq_ef_f32(square.data_ptr(), err.data_ptr(), q.data_ptr(), p.data_ptr(), side, side, rank,
                                      ws_ptr, ws_len, stream)
    else:
        rc = lib.conef_psgd_mq_f32(square.data_ptr(), q.data_ptr(), p.data_ptr(), side, side, rank, ws_ptr, ws_len,
                                   stream)
    _lib.check(rc, "conef_psgd_mq")
    _lib.check(lib.conef_gram_schmidt_f32(p.data_ptr(), side, rank, eps, ws_ptr, ws_len, stream),
               "conef_gram_schmidt_f32")
    _lib.check(lib.conef_psgd_mtp_f32(square.data_ptr(), p.data_ptr(), q.data_ptr(), side, side, rank, ws_ptr, ws_len,
                                      stream), "conef_psgd_mtp_f32")
    if err is not None:
        rc = lib.conef_psgd_pqt_ef_f32(square.data_ptr(), err.data_ptr(), p.data_ptr(), q.data_ptr(), side, side, rank,
                                       stream)
    else:
        rc = lib.conef_psgd_pqt_f32(square.data_ptr(), p.data_ptr(), q.data_ptr(), side, side, rank, stream)
    _lib.check(rc, "conef_psgd_pqt")
    if square is not input_tensor:
        input_tensor.copy_(square[:total_length])
    if not state.warm_start:
        state.p_memory_dict.clear()
        state.q_memory_dict.clear()
    state.maybe_increase_iter(bucket)
    return _bucket.completed_future(input_tensor)
