"""One-GPU offloading runtime for routed experts (reference: ferry/runtime.py).

Per MoE layer call (world = 1):
  1. history: the device window counters of the layer are updated from ``selected``; the
     same kernel writes the expert IDs (uint8; of a large call each expert's demand instead) and
     the layer's scores straight into mapped host memory -- the host must know the misses to
     enqueue fetches;
  2. the layout kernel is enqueued before the host waits for those results, so it overlaps
     the host planning;
  3. the C++ planner picks the misses (ascending expert) and their slots (routing-aware
     eviction, bit-exact with the reference) and the H2D engine enqueues their copies on its
     own stream;
  4. the misses are copied with ``hipMemcpyAsync`` on the fetch engine's DMA streams while the
     experts already resident run; the compute stream then waits on the GPU for the copies and
     runs the fetched experts.  A prefill-sized call copies its misses in a few groups,
     heaviest expert first, each computed as soon as its copies land, so that only the
     lightest group's compute is left after the last copy; a decode-sized call runs all its
     misses in one launch after the last copy (``split_fetch=True``, with packed rows: one
     launch per sub-batch as the engine unpacks it).  ``overlap=False`` restores the
     reference's serial host wait.  ``copy='kernel'`` (not the reference's scheme) copies a
     decode-sized call's misses with one copy-kernel launch on the compute stream instead and
     then runs every active expert in one FFN launch: no idle link between copies and no
     cross-queue wait, but no overlap either (the copy kernel's host reads slow the HBM-bound
     kernels that run beside it, so nothing runs beside it);
  5. the combine kernel sums each token's k expert rows in fp32 (ascending expert ID).

The one-launch decode FFN bounds its cross-workgroup wait; a wait that gives up leaves rows
unwritten and counts a timeout on the device.  The history kernel copies that count next to the
routing IDs, so the next call raises RuntimeError when it grew (an earlier call's output is then
invalid), and so do ``reset`` and ``close``.
"""
import ctypes
import time

import numpy as np
import torch
import torch.distributed as dist

from . import expert_ops as ops
from ._lib import check, lib
from .h2d import DMA, KERNEL
from .hostmem import mapped_buffer
from .metadata import DeviceGateHistory, GateHistory, RouteGather
from .policy import Controller
from .transport import Transport


# A layer call with at least this many (token, expert) pairs fetches its misses in up to CHUNKS
# groups, heaviest first, and computes each group as soon as its copies land.  Decode calls
# (few pairs, little compute per expert) keep one group and one launch for their misses: with
# packed rows, one launch per unpacked sub-batch (OffloadRuntime(split_fetch=True)) shortens
# the step by about 1 % but adds a launch's fixed cost of GPU time for each.
CHUNK_MIN_PAIRS = 16384
CHUNKS = 6
# Packed chunked calls: CUs that the tiled kernels leave to the unpacking of the rows still being
# copied.  A tiled workgroup holds its CU's registers for the whole launch, so without them a row's
# unpacking, and the copies behind it, wait for a launch to end: 26 DeepSeek-V2-Lite layers of 65,536
# tokens, every expert fetched, take 372.5 ms with 0, 362.7 with 8, 362.2 with 16, 360.7 with 32 (FFN
# 7.7, 7.9, 8.1, 8.3 ms a layer, which the copies of 13.2 ms hide); 48 Qwen3 layers of 8192 tokens
# 703.1, 703.5, 702.9 and 701.5.
UNPACK_CUS = 16

# A call with at least this many pairs has the device check its IDs and count each expert's demand
# instead of the host planner, for which the GPU waits: from launch to plan 512 tokens x 8 of 128
# took 25.4 us with the IDs and 24.2 with the counts, 8192 x 8 53 and 29, 256 x 8 23.7 and 23.2
# (about the same), 16 x 8 22.3 and 23.1.
COUNT_MIN_PAIRS = 2048


def expert_ops():
    """The native op module (reference: ferry/runtime.py:26-31)."""
    return ops


class _LayerLists:
    """Buffers of ferry_layer_lists and their addresses: 0 the active experts, 1 the resident, 2
    the fetched ones."""

    def __init__(self, experts):
        self.experts = experts
        self.slot_of = np.empty(experts, np.int32)
        self.lists = np.empty((3, 2, experts), np.int32)
        self.slots = np.empty((3, experts), np.int64)
        self.sizes_array = np.zeros(9, np.int64)
        self.sizes = [0] * 9
        self.slot_of_ptr, self.lists_ptr = self.slot_of.ctypes.data, self.lists.ctypes.data
        self.slots_ptr, self.sizes_ptr = self.slots.ctypes.data, self.sizes_array.ctypes.data

    def slots_at(self, which):
        return self.slots_ptr + 8 * which * self.experts

    def entry(self, which):
        """(experts, row counts, entries, most rows, least rows) of one list."""
        at = self.lists_ptr + 8 * which * self.experts
        n, most, least = self.sizes[3 * which:3 * which + 3]
        return at, at + 4 * self.experts, n, most, least


class OffloadRuntime:
    def __init__(self, spec, pool, capacities, policy, topology, history_window=128,
                 balance_tol_bps=200, salt=1, eviction_score='frequency', overlap=True,
                 timing=False, copy='dma', pack=False, pack_threads=16, split_fetch=False):
        if dist.is_available() and dist.is_initialized() and dist.get_world_size() != 1:
            raise NotImplementedError('ferry_amd runs on one GPU (world = 1)')
        if len(capacities) != 1:
            raise NotImplementedError('ferry_amd runs on one GPU (world = 1)')
        self.spec = spec
        self.pool = pool
        self.rank, self.world = 0, 1
        self.capacities = capacities
        self.cap = capacities[0]
        self.window = history_window
        self.overlap = overlap
        self.timing = timing
        if copy not in ('dma', 'kernel'):
            raise ValueError("copy must be 'dma' or 'kernel'")
        self.copy = copy
        # packed decode calls: compute the fetched experts sub-batch by sub-batch as the engine
        # unpacks them (one FFN launch per sub-batch) instead of in one launch after the last
        self.split_fetch = bool(split_fetch)
        # a lossless packed copy of the pool for the host link, made once; every engine of this
        # runtime fetches packed rows in DMA mode and unpacks them on the GPU
        # (pack: True, or a PackedPool of this pool built by the caller and shared; ``pool``
        # itself may be a PackedPool, whose engines need no raw pool)
        from .h2d import PackedPool
        self.packed = None
        if isinstance(pool, PackedPool):
            self.packed = pool
        elif pack is not None and pack is not False:
            self.packed = pack if isinstance(pack, PackedPool) else PackedPool(pool, pack_threads)
        self.ops = expert_ops()
        self.device = torch.device('cuda', torch.cuda.current_device())
        self.cache = torch.empty((self.cap, spec.expert_elements), dtype=torch.bfloat16,
                                 device=self.device)
        self.controller = Controller(spec, capacities, policy, topology, balance_tol_bps, salt)
        self.gather = RouteGather(spec.topk, spec.experts, history_window, eviction_score)
        self.transport = Transport(self.ops, spec.topk, spec.experts)
        # mapped host staging: [scores f32 E | IDs u8 T*k or demand records i32], and
        # [timeouts i32 | ready i32 ...]
        self._stage_host = None
        self._ready_host = None
        self._bufs = {}
        self._lists = _LayerLists(spec.experts)
        self._ready_seq = 0
        # calls wait for their routing IDs by polling the history kernel's ready words (False:
        # on the event recorded after that kernel)
        self._poll_ids = True
        self.h2d = None
        self.reset()

    # -- state -------------------------------------------------------------------------------

    def reset(self):
        """Empty expert cache and routing history (start of every measured run).  Raises
        RuntimeError (after the reset) if a decode FFN wait gave up since the last check."""
        self._flush_used()
        if self.h2d is not None:
            self.h2d.synchronize()
        torch.cuda.synchronize(self.device)
        late = self._timeouts_since_check()
        self.controller.reset()
        spec = self.spec
        self.history = GateHistory(spec.layers, spec.experts, self.window)
        self.device_history = DeviceGateHistory(spec.layers, spec.experts, spec.topk, self.window,
                                                self.device)
        # the engine is reset in place rather than rebuilt: a new engine's streams can land on
        # the hardware queue of this runtime's compute stream and serialise with it
        if self.h2d is not None:
            self.h2d.reset()
        elif self.packed is not None:
            self.h2d = self.ops.H2DEngine.from_packed(self.cache, self.packed)
        else:
            self.h2d = self.ops.H2DEngine(self.cache, self.pool)
        self._kernel_copy = self.copy == 'kernel' and self.h2d.kernel_ok
        self._defer_last = False
        if self.copy == 'kernel' and not self._kernel_copy:
            raise RuntimeError("copy='kernel' needs a device-mapped pool with 16-byte rows")
        self._copy_mode = None
        self.event = 0
        self.fetches_per_rank = np.zeros(self.world, np.int64)
        self.decode_fetches_per_rank = np.zeros(self.world, np.int64)
        self.serial_wait_ns = 0
        self.timings = []
        self.step_marks = []   # timing=True: (ids ready, copies queued, copies done, compute resumes)
        self.kernel_bytes = dict(up=0, down=0, flops=0, experts=0, launches=0)
        # host time per phase of execute (ns, timing=True): the planning path between the
        # wait for the routing IDs and the fetch enqueue is on the critical path of a step
        self.host_ns = dict(enqueue_before_wait=0, wait_for_ids=0, plan=0, fetch_enqueue=0,
                            enqueue_after_fetch=0)
        if late:
            raise RuntimeError(self._timeout_message(late))

    # -- decode FFN timeouts -----------------------------------------------------------------

    def _timeouts_since_check(self):
        """Device-wide decode FFN timeouts counted since the last check (reads the device)."""
        now = self.ops.ffn_sync_timeouts()
        seen = getattr(self, '_timeouts_seen', now)
        self._timeouts_seen = now
        return now - seen

    @staticmethod
    def _timeout_message(n):
        return (f'{n} wait(s) of the one-launch decode FFN gave up on this device: the rows of '
                f'those experts were not written, so the output of an earlier layer call is '
                f'invalid')

    def _buffers(self, tokens):
        b = self._bufs.get(tokens)
        if b is None:
            spec, k = self.spec, self.spec.topk
            b = dict(act=torch.empty((tokens * k, spec.intermediate), dtype=torch.bfloat16,
                                     device=self.device),
                     part=torch.empty((tokens * k, spec.hidden), dtype=torch.bfloat16,
                                      device=self.device),
                     layout=None)
            # a large call plans from demand records instead of IDs (frequency scores only)
            b['stage'] = tokens * k
            b['ready_n'] = b['ready_counted'] = self.ops.history_ready_words(tokens, k)
            b['counted'] = tokens * k >= COUNT_MIN_PAIRS
            if b['counted']:
                blocks = self.ops.history_count_blocks(tokens)
                b['stage'] = max(b['stage'], 4 * blocks * self.ops.history_count_words(spec.experts))
                b['ready_counted'] = 1 + blocks
            self._bufs[tokens] = b
        # coherent mapped host memory: the history kernel writes the layer's scores, the uint8 IDs
        # or demand records, the timeout count and its ready words straight into it, so the host
        # needs no D2H copy.  The timeout word and the ready words have a buffer of their own, in
        # which no other data of an earlier call can look like this call's number.
        n = 4 * self.spec.experts + b['stage']
        if self._stage_host is None or self._stage_host.numel() < n:
            self._stage_host, self._stage_ptr = mapped_buffer(max(n, 4096))
        n = 4 + 4 * max(b['ready_n'], b['ready_counted'])
        if self._ready_host is None or self._ready_host.numel() < n:
            self._ready_host, self._ready_ptr = mapped_buffer(max(n, 4096))
            self._ready_host.zero_()   # no call's number
            self._ready_host_ptr = self._ready_host.data_ptr()
            # int32 view for the timeout word (read right after the routing readback, on the
            # path to the first copy: a torch slice and view there cost about 10 us)
            self._ready_i32 = self._ready_host.numpy().view(np.int32)
        return b

    # -- one layer call ------------------------------------------------------------------------

    def execute(self, layer, hidden, selected, weights, probs_tail, shared=None):
        """One MoE layer call (runtime.py:64-89).  ``shared`` (an ``expert_ops.SharedExpert``,
        not a reference argument) adds an always-on expert's output to every token, as
        DeepSeek-V2's block does after the routed experts; it runs while the misses copy."""
        t_enter = time.perf_counter_ns()
        spec = self.spec
        T, k = selected.shape
        E = spec.experts
        if hidden.dtype != torch.bfloat16 or hidden.dim() != 2 or hidden.shape[1] != spec.hidden:
            raise RuntimeError('hidden must be bf16 [tokens, hidden]')
        if not hidden.is_cuda:
            raise RuntimeError('hidden must be a CUDA tensor')
        hidden = hidden.contiguous()
        stream = torch.cuda.current_stream(self.device)
        handle = stream.cuda_stream
        buf = self._buffers(T)
        selected = selected.contiguous()
        weights = weights.to(torch.bfloat16).contiguous()

        # 1. history; the kernel writes scores, IDs and the device's decode FFN timeout count
        # into the mapped host staging buffer (with probability scores its scores go unused)
        frequency = self.gather.score == 'frequency'
        counted = frequency and buf['counted']
        # the ready words after the timeout word carry this call's number once the kernel's
        # host-memory writes are visible
        self._ready_seq = self._ready_seq % 0x7FFFFFFF + 1
        seq = self._ready_seq
        staged = self._stage_ptr + 4 * E
        self.device_history.update(layer, selected, self._stage_ptr, None if counted else staged,
                                   self._ready_ptr, self._ready_ptr + 4, seq,
                                   staged if counted else None)
        tail_host = None
        if not frequency:
            tail = min(T, self.window)
            tail_host = probs_tail[-tail:].float().to('cpu', non_blocking=True)
        if self.timing:
            # timestamp of the routing IDs (the history kernel's end) for critical_path_timing
            d2h = torch.cuda.Event(enable_timing=True)
            d2h.record(stream)
        # one event both releases the IDs to the host and marks the slots that the previous call
        # read on this stream (no event of their own between that call's kernels)
        pend = self._pending_used
        if pend is not None and pend[1] != handle:
            self._flush_used()
            pend = None
        self._pending_used = None
        ids_event = self.h2d.mark_used_record(pend[0] if pend is not None else [], stream)

        # 2. layout (overlaps the host planning)
        buf['layout'] = self.ops.layout(selected, weights, E, out=buf['layout'])
        lay = buf['layout']
        chunked = T * k >= CHUNK_MIN_PAIRS
        on_stream = self.overlap and not chunked and self._kernel_copy
        # packed decode calls: the last sub-batch's unpack runs on this stream right after the
        # copies (one cross-queue wait before the fetched experts, not two)
        defer = (self.packed is not None and self.overlap and not chunked and not on_stream
                 and not self.timing)
        if defer != self._defer_last:
            self.h2d.defer_last = defer
            self._defer_last = defer

        # 3. plan + fetch
        t_sync = time.perf_counter_ns()
        if self._poll_ids:
            # poll the history kernel's ready words: they are seen about 5 us before the event's
            # wait returns, and they show the previous call's slot reads complete
            self.h2d.wait_ready(ids_event, self._ready_host_ptr + 4,
                                buf['ready_counted' if counted else 'ready_n'], seq)
        else:
            self.h2d.event_synchronize(ids_event)
        t_ready = time.perf_counter_ns()
        count = int(self._ready_i32[0])
        if count != self._timeouts_seen:
            late, self._timeouts_seen = count - self._timeouts_seen, count
            raise RuntimeError(self._timeout_message(late))
        self._set_copy_mode(on_stream, stream)
        # with chunks or timing the copies are queued here; otherwise the planner's native call
        # queues them itself, right after planning
        queue_here = chunked or self.timing
        if counted:
            fetches, counts = self.controller.plan_fetch_counts(
                self.event, layer, staged, T, self._stage_ptr,
                None if queue_here else self.h2d.handle)
        elif frequency:
            fetches, counts = self.controller.plan_fetch(
                self.event, layer, staged, T, k, self._stage_ptr,
                None if queue_here else self.h2d.handle)
        else:
            self.history.update(layer, tail_host.numpy())
            scores = self.history.scores(layer)
            ids = self._stage_host.numpy()[4 * E:4 * E + T * k].astype(np.int64).reshape(T, k)
            fetches, _, counts = self.controller.plan(self.event, layer, ids, np.zeros(T, np.int64),
                                                      scores)
            queue_here = True
        t_plan = time.perf_counter_ns()
        demand = self.controller.demand if frequency else np.bincount(ids.reshape(-1), minlength=E)
        lists = self._layer_lists(layer, demand, fetches)
        missing_keys = None
        # copy order: heaviest expert first, so that the compute left after the last copy is
        # the lightest (the planner's slot choices do not depend on the order of the copies)
        if chunked and len(fetches) > 1:
            missing_keys = fetches[:, 1] - layer * E
            order = np.argsort(-demand[missing_keys], kind='stable')
            groups = [g for g in np.array_split(order, min(CHUNKS, len(fetches))) if len(g)]
        else:
            groups = [np.arange(len(fetches))] if queue_here else [None]
        timing = self.timing and len(fetches) > 0
        if timing:
            copy_stream = stream if on_stream else self.h2d.stream
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ev[0].record(copy_stream)
        if queue_here and len(fetches):
            for g in groups:
                self.h2d.fetch(fetches[g, 2], fetches[g, 1])
        if (self.split_fetch and not chunked and not on_stream and self.packed is not None
                and len(fetches) > 1):
            # each sub-batch's experts run as soon as the engine has unpacked it, so only the
            # last sub-batch's experts follow the call's last copy
            ends = self.h2d.groups()
            if len(ends) > 1:
                missing_keys = fetches[:, 1] - layer * E
                groups = [np.arange(a, b) for a, b in zip([0] + ends[:-1], ends)]
        t_fetch = time.perf_counter_ns()
        if timing:
            ev[1].record(copy_stream)

        # 4. experts: resident first, then the fetched ones (chunk by chunk as they land)
        common = (hidden, lay, buf, T, k, handle)
        # CUs that the tiled kernels leave to the unpacking of rows still being copied (without
        # overlap the call waits for all of them before its first expert)
        spare = (UNPACK_CUS if chunked and self.overlap and self.packed is not None and len(fetches)
                 else 0)
        n_active, n_resident = lists.sizes[0], lists.sizes[3]
        if not self.timing:
            # the reads below are marked by the next call's ID event on this stream (or by
            # _flush_used); set before they are queued, so that a call that fails part-way still
            # orders later copies into these slots after whatever it queued
            self._pending_used = (lists.slots[0][:n_active].copy(), handle, stream)
        if not self.overlap and len(fetches):
            started = time.perf_counter_ns()
            self.h2d.wait_host(fetches[:, 2])
            self.serial_wait_ns += time.perf_counter_ns() - started
        mark = self.ops.timing_mark() if timing else 0
        waits = []
        if on_stream:
            # the copies are queued on this stream (the wait on their events costs nothing);
            # resident rows may come from DMA copies of earlier calls
            self.h2d.wait_stream_at(lists.slots_at(0), n_active, handle)
            if timing:
                waits.append((ev[0], ev[1]))   # the copy kernel holds this stream
            self._ffn(common, *lists.entry(0))
        elif n_resident:
            self.h2d.wait_stream_at(lists.slots_at(1), n_resident, handle)
            self._ffn(common, *lists.entry(1), spare)
        shared_out = None
        if shared is not None:
            out = self._shared_out(T)
            shared_out = shared(hidden, out=out, spare_cus=spare) if spare else shared(hidden, out=out)
        if len(fetches) and not on_stream:
            for g in groups:
                w0 = w1 = None
                if timing:
                    w0 = torch.cuda.Event(enable_timing=True)
                    w0.record(stream)
                if len(groups) == 1:
                    self.h2d.wait_stream_at(lists.slots_at(2), len(fetches), handle)
                else:
                    self.h2d.wait_stream(fetches[g, 2], stream)
                if timing:
                    w1 = torch.cuda.Event(enable_timing=True)
                    w1.record(stream)
                    waits.append((w0, w1))
                if len(groups) == 1:
                    self._ffn(common, *lists.entry(2))
                else:
                    el = np.sort(missing_keys[g])
                    rows = demand[el]
                    self._ffn(common, el.astype(np.int32).tobytes(), rows.astype(np.int32).tobytes(),
                              len(el), int(rows.max()), int(rows.min()),
                              spare if g is not groups[-1] else 0)
        if self.timing:
            self.h2d.mark_used(lists.slots[0][:n_active], stream)
        if timing:
            self.timings.append((ev, waits, (mark, self.ops.timing_mark())))
            self.step_marks.append((d2h, ev[0], ev[1], waits[-1][1] if waits else None))
        self.fetches_per_rank += counts
        if self.event >= spec.layers:
            self.decode_fetches_per_rank += counts
        self.event += 1

        # 5. combine (+ the shared experts' output)
        out = self.ops.combine(buf['part'], T, k, spec.hidden, addend=shared_out)
        if self.timing:
            h = self.host_ns
            h['enqueue_before_wait'] += t_sync - t_enter
            h['wait_for_ids'] += t_ready - t_sync
            h['plan'] += t_plan - t_ready       # with frequency scores: plan + fetch enqueue
            h['fetch_enqueue'] += t_fetch - t_plan
            h['enqueue_after_fetch'] += time.perf_counter_ns() - t_fetch
        return out

    def _flush_used(self):
        """Mark the slots of the last call as read, with an event of their own."""
        pend = getattr(self, '_pending_used', None)
        if pend is not None and self.h2d is not None:
            self.h2d.mark_used(pend[0], pend[2])
        self._pending_used = None

    def _set_copy_mode(self, on_stream, stream):
        """Copy kernel on ``stream`` for on-stream calls, DMA copies otherwise."""
        mode = (on_stream, stream.cuda_stream if on_stream else None)
        if mode != self._copy_mode:
            self.h2d.engine = KERNEL if on_stream else DMA
            self.h2d.set_kernel_stream(stream if on_stream else None)
            self._copy_mode = mode

    def _shared_out(self, tokens):
        b = self._bufs[tokens]
        if 'shared' not in b:
            b['shared'] = torch.empty((tokens, self.spec.hidden), dtype=torch.bfloat16,
                                      device=self.device)
        return b['shared']

    def _layer_lists(self, layer, demand, fetches):
        """The call's expert lists (ferry_layer_lists) in this runtime's buffers, which the native
        calls of the same layer call read."""
        lists, ctl = self._lists, self.controller
        check(lib().ferry_layer_lists(ctl._slots_ptr, self.cap, layer, self.spec.experts,
                                      demand.tobytes(), fetches.tobytes(), len(fetches),
                                      lists.slot_of_ptr, lists.lists_ptr, lists.slots_ptr,
                                      lists.sizes_ptr), 'layer_lists')
        lists.sizes = lists.sizes_array.tolist()
        return lists

    def _ffn(self, common, expert_list, list_rows, n, most, least, spare=0):
        """Phase 1 (gate/up + SwiGLU) and phase 2 (down + weight) for the ``n`` experts of
        ``expert_list`` with ``list_rows`` rows each (int32, host addresses or bytes)."""
        hidden, lay, buf, T, k, handle = common
        spec = self.spec
        check(lib().ferry_expert_ffn_spare(
            self.cache.data_ptr(), self.cap, spec.hidden, spec.intermediate, hidden.data_ptr(), T, k,
            lay.w_sorted.data_ptr(), lay.starts.data_ptr(), lay.rows.data_ptr(),
            lay.cols.data_ptr(), expert_list, n, self._lists.slot_of_ptr, spec.experts, most, least,
            list_rows, buf['act'].data_ptr(), buf['part'].data_ptr(), 0, self.ops.PHASE_BOTH,
            spare, handle), 'expert_ffn')
        if self.timing:
            H, I = spec.hidden, spec.intermediate
            data = (list_rows if isinstance(list_rows, bytes)
                    else ctypes.string_at(list_rows, 4 * n))
            rows = int(np.frombuffer(data, np.int32).sum())
            d = n
            # algorithmic bytes: weights read once, x / activation rows read, outputs written
            self.kernel_bytes['up'] += d * 2 * I * H * 2 + rows * (H * 2 + I * 2)
            self.kernel_bytes['down'] += d * H * I * 2 + rows * (I * 2 + H * 2 + 2)
            self.kernel_bytes['flops'] += 2 * 3 * H * I * rows
            self.kernel_bytes['experts'] += d
            self.kernel_bytes['launches'] += 1

    def fetch_timing(self):
        """(total fetch ms, exposed wait ms, overlapped compute ms) over the layer calls recorded
        with timing=True.  fetch: first copy start to last copy end on the copy stream.  exposed:
        how long the compute stream stalled on the copies.  overlapped: the time, inside each
        call's fetch window, covered by the compute kernels of that call (resident experts,
        shared experts, and missing experts whose copies landed early); it needs the library's
        per-launch timing (expert_ops.timing_enable)."""
        torch.cuda.synchronize(self.device)
        fetch = exposed = overlapped = 0.0
        for ev, waits, (m0, m1) in self.timings:
            fetch += ev[0].elapsed_time(ev[1])
            exposed += sum(max(0.0, a.elapsed_time(b)) for a, b in waits)
            overlapped += self.ops.timing_overlap(m0, m1, ev[0], ev[1])
        return fetch, exposed, overlapped

    def critical_path_timing(self):
        """Mean GPU-side gaps (ms) over the calls with copies recorded with timing=True: from the
        routing IDs being written (the history kernel's end) to the copies being queued (the
        host reads the IDs and plans in between), and from the last copy's end to the compute
        stream resuming after its wait for the copies."""
        torch.cuda.synchronize(self.device)
        plan, resume = [], []
        for d2h, q, done, w1 in self.step_marks:
            plan.append(d2h.elapsed_time(q))
            if w1 is not None:
                resume.append(done.elapsed_time(w1))
        mean = lambda v: sum(v) / len(v) if v else None   # noqa: E731
        return dict(ids_to_copy_queue_ms=mean(plan), copy_end_to_compute_ms=mean(resume),
                    calls=len(plan))

    def close(self):
        """Drain the runtime's work; raises RuntimeError if a decode FFN wait gave up since the
        last check."""
        self._flush_used()
        if self.h2d is not None:
            self.h2d.synchronize()
        torch.cuda.synchronize(self.device)
        late = self._timeouts_since_check()
        if late:
            raise RuntimeError(self._timeout_message(late))
