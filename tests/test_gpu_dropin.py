"""The reference runtime's own call order, driven through ferry_amd's drop-in names.

FERRY's ``OffloadRuntime.execute`` (ferry/runtime.py:64-89) makes these calls per MoE layer:
RouteGather.collect -> GateHistory.update / scores -> Controller.plan -> H2DEngine.fetch ->
layer_slots -> device_layout -> Transport.dispatch (pack_dispatch -> exchange ->
unpack_dispatch) -> H2DEngine.wait_host -> execute_experts -> H2DEngine.mark_used ->
Transport.combine (reduce_partials -> exchange -> scatter_returned).  ``ReferenceOrder`` below
makes exactly those calls on ferry_amd's modules, which is what a FERRY runtime does once its
imports point at them.  Over a sequence of layer calls that forces evictions, its outputs and
eviction state must equal ferry_amd's fused runtime bit for bit, and the outputs must match the
oracle.  Each step's bytes and indices are checked against the oracle separately.
"""
import numpy as np
import pytest
import torch

from oracle.experts import execute_experts_ref, moe_layer_ref, reduce_partials_ref
from oracle.layout import layout_closed_form
from oracle.transport import pack_dispatch_ref, packets_closed_form, unpack_dispatch_ref

pytestmark = pytest.mark.gpu


class ReferenceOrder:
    """The steps of ferry/runtime.py:35-89 on ferry_amd's API mirrors (world = 1)."""

    def __init__(self, spec, pool, cap, window=128):
        from ferry_amd.metadata import GateHistory, RouteGather
        from ferry_amd.policy import Controller
        from ferry_amd.quota import Topology
        from ferry_amd.runtime import expert_ops
        from ferry_amd.transport import Transport
        self.spec, self.cap = spec, cap
        self.ops = expert_ops()
        self.cache = torch.empty((cap, spec.expert_elements), dtype=torch.bfloat16, device='cuda')
        self.controller = Controller(spec, [cap], 'ferry', Topology.uniform(1, spec.experts))
        self.gather = RouteGather(spec.topk, spec.experts, window, 'frequency')
        self.transport = Transport(self.ops, spec.topk, spec.experts)
        self.history = GateHistory(spec.layers, spec.experts, window)
        self.h2d = self.ops.H2DEngine(self.cache, pool)
        self.event = 0
        self.last_fetches = None

    def execute(self, layer, hidden, selected, weights, probs_tail):
        from ferry_amd.layout import device_layout
        from ferry_amd.policy import layer_slots
        spec = self.spec
        ids, origins, tail = self.gather.collect(selected, probs_tail)
        self.history.update(layer, tail)
        fetches, destinations, counts = self.controller.plan(
            self.event, layer, ids, origins, self.history.scores(layer))
        mine = fetches[fetches[:, 0] == 0]
        fetch_slots = mine[:, 2].tolist()
        self.h2d.fetch(fetch_slots, mine[:, 1].tolist())
        slot_of = layer_slots(self.controller.slots[0], self.cap, layer, spec.experts)
        layout = device_layout(ids, destinations, selected.shape[0], 0, spec.experts, slot_of)
        received, received_weights = self.transport.dispatch(hidden, selected, weights, layout)
        self.h2d.wait_host(fetch_slots)
        self.last_fetches = mine
        groups = layout['groups']
        slots = [g[3] for g in groups]
        parts = self.ops.execute_experts(self.cache, received, received_weights, slots,
                                         [g[1] for g in groups], [g[2] for g in groups],
                                         spec.hidden, spec.intermediate)
        self.h2d.mark_used(slots)
        self.event += 1
        return self.transport.combine(hidden, parts, layout)


def _routing(T, E, k, pool_size, rng):
    """Each token picks k distinct experts among a per-call subset of ``pool_size`` experts."""
    subset = rng.choice(E, pool_size, replace=False)
    sel = np.stack([rng.choice(subset, k, replace=False) for _ in range(T)]).astype(np.int64)
    logits = rng.standard_normal((T, k)).astype(np.float32)
    w = torch.softmax(torch.from_numpy(logits), -1).to(torch.bfloat16)
    return torch.from_numpy(sel), w


def test_reference_order_matches_fused_runtime(device):
    """Two layers, a 12-slot cache and 10 active experts per call: misses, evictions, slot
    reuse (WAR through mark_used) and calls that take the skinny, mid and tiled kernels."""
    from ferry_amd import workloads
    from ferry_amd.model import ModelSpec
    from ferry_amd.quota import Topology
    from ferry_amd.runtime import OffloadRuntime
    spec = ModelSpec('qwen3_moe', (0, 1), 32, 4, 256, 128)
    E, k, H, I, cap = spec.experts, spec.topk, spec.hidden, spec.intermediate, 12
    pool = workloads.make_pool(spec, spec.layers, seed=5)
    ref = ReferenceOrder(spec, pool, cap)
    fused = OffloadRuntime(spec, pool, [cap], 'ferry', Topology.uniform(1, E))
    rng = np.random.default_rng(11)
    g = torch.Generator().manual_seed(12)
    copies = 0
    for call, T in enumerate([16, 3, 300, 1, 64, 16, 129, 40, 16, 2]):
        layer = call % 2
        print(f'call {call}: layer {layer}, {T} tokens', flush=True)
        sel, w = _routing(T, E, k, 10, rng)
        x = torch.randn((T, H), generator=g).to(torch.bfloat16)
        xd, seld, wd = x.to(device), sel.to(device), w.to(device)
        out_ref = ref.execute(layer, xd, seld, wd, None)
        # after wait_host every fetched slot holds its pool row
        for _, key, slot in ref.last_fetches:
            assert torch.equal(ref.cache[slot].cpu(), pool[key]), (call, key, slot)
        copies += len(ref.last_fetches)
        out_fused = fused.execute(layer, xd, seld, wd, None)
        torch.cuda.synchronize()
        assert torch.equal(out_ref, out_fused), f'call {call}'
        for a, b in ((ref.controller.slots, fused.controller.slots),
                     (ref.controller.owner, fused.controller.owner),
                     (ref.controller.last, fused.controller.last)):
            assert np.array_equal(a, b), f'call {call}'
        oracle = moe_layer_ref(lambda e: pool[layer * E + e], x, sel, w, E, H, I)
        torch.testing.assert_close(out_ref.cpu().float(), oracle.float(), rtol=2e-2, atol=1e-2)
    assert ref.h2d.copies == fused.h2d.copies == copies
    assert copies > cap                 # the sequence evicted
    assert ref.transport.dispatch_bytes == ref.transport.combine_bytes == 0
    ref.h2d.synchronize()
    fused.close()


@pytest.mark.parametrize('T,E,k,H,I', [(40, 16, 4, 256, 128), (300, 64, 6, 512, 256)])
def test_dispatch_combine_steps_bit_exact(device, T, E, k, H, I):
    """device_layout, pack_dispatch, unpack_dispatch, execute_experts, reduce_partials and
    scatter_returned one by one against the oracle: bytes and indices bit-exact, expert rows
    within rel 2e-2 / abs 1e-2, the fp32 sums bit-exact on the same expert rows."""
    from ferry_amd import expert_ops as ops
    from ferry_amd.layout import device_layout
    rng = np.random.default_rng(T)
    g = torch.Generator().manual_seed(T)
    sel, w = _routing(T, E, k, E, rng)
    x = torch.randn((T, H), generator=g).to(torch.bfloat16)
    rows_w = (torch.randn((E, 3 * H * I), generator=g) * 0.02).to(torch.bfloat16)
    slot_of = rng.permutation(E)
    cache = torch.empty_like(rows_w)
    cache[torch.from_numpy(slot_of)] = rows_w
    cache = cache.to(device)

    layout = device_layout(sel.numpy(), np.zeros((T, k), np.int64), T, 0, E, slot_of)
    ref_lay = layout_closed_form(sel.numpy(), E, w.view(torch.int16).numpy())
    assert torch.equal(layout['send_idx'].cpu(), torch.arange(T))
    assert np.array_equal(layout['send_ids'].cpu().numpy(), ref_lay['send_ids'])
    assert layout['send_counts'] == layout['recv_counts'] == [T]
    groups = layout['groups']
    assert [g_[0] for g_ in groups] == [e for e in range(E) if ref_lay['counts'][e]]
    for e, r, c, slot in groups:
        a, b = ref_lay['starts'][e], ref_lay['starts'][e + 1]
        assert np.array_equal(r.cpu().numpy(), ref_lay['rows'][a:b])
        assert np.array_equal(c.cpu().numpy(), ref_lay['cols'][a:b])
        assert slot == slot_of[e]

    payload = ops.pack_dispatch(x.to(device), sel.to(device), w.to(device), layout['send_idx'],
                                layout['send_ids'], E)
    want = pack_dispatch_ref(x, sel, w, torch.arange(T), torch.from_numpy(ref_lay['send_ids']), E)
    assert torch.equal(payload.cpu(), want)
    assert np.array_equal(want.numpy(), packets_closed_form(x, ref_lay['send_ids'], ref_lay['w_sorted']))
    received, rweights = ops.unpack_dispatch(payload, H, k)
    ux, uw = unpack_dispatch_ref(want, H, k)
    assert torch.equal(received.cpu(), ux) and torch.equal(rweights.cpu(), uw)

    parts = ops.execute_experts(cache, received, rweights, [g_[3] for g_ in groups],
                                [g_[1] for g_ in groups], [g_[2] for g_ in groups], H, I)
    rows = [torch.from_numpy(ref_lay['rows'][ref_lay['starts'][e]:ref_lay['starts'][e + 1]])
            for e, _, _, _ in groups]
    cols = [torch.from_numpy(ref_lay['cols'][ref_lay['starts'][e]:ref_lay['starts'][e + 1]])
            for e, _, _, _ in groups]
    want_parts = execute_experts_ref([rows_w[e] for e, _, _, _ in groups], ux, uw, rows, cols, H, I)
    for got, exp in zip(parts, want_parts):
        torch.testing.assert_close(got.cpu().float(), exp.float(), rtol=2e-2, atol=1e-2)

    partial = ops.reduce_partials(parts, [g_[1] for g_ in groups], T, H, x.to(device))
    assert torch.equal(partial.cpu(), reduce_partials_ref([p.cpu() for p in parts], rows, T, H))
    back = ops.scatter_returned(partial, layout['send_idx'], T)
    assert torch.equal(back, partial)   # world = 1: an fp32 round trip of every row
    oracle = moe_layer_ref(lambda e: rows_w[e], x, sel, w, E, H, I)
    torch.testing.assert_close(back.cpu().float(), oracle.float(), rtol=2e-2, atol=1e-2)


@pytest.mark.parametrize('T,H,k', [(3, 64, 1), (5, 256, 2), (7, 256, 3), (65, 512, 4), (9, 2048, 6),
                                   (33, 2048, 8), (4, 20, 5)])
def test_packets_of_every_alignment(device, T, H, k):
    """Packet pitches 2H + 3k that are odd and multiples of 2, 4, 8 and 16, a payload that starts at
    an odd address, hidden rows that are no multiple of 16 bytes: packets bit-equal to the closed
    form, and split back into the same rows and weights."""
    from ferry_amd import expert_ops as ops
    from ferry_amd._lib import last_error, lib
    rng = np.random.default_rng(T * H + k)
    E = 4 * k
    sel, w = _routing(T, E, k, E, rng)
    x = torch.randn((T, H), generator=torch.Generator().manual_seed(k)).to(torch.bfloat16)
    ref = layout_closed_form(sel.numpy(), E, w.view(torch.int16).numpy())
    want = torch.from_numpy(packets_closed_form(x, ref['send_ids'], ref['w_sorted']))
    xd, seld, wd = x.to(device), sel.to(device), w.to(device)
    idx, ids = torch.arange(T, device=device), torch.from_numpy(ref['send_ids']).to(device)
    payload = ops.pack_dispatch(xd, seld, wd, idx, ids, E)
    assert torch.equal(payload.cpu(), want)
    pitch = 2 * H + 3 * k
    flat = torch.full((T * pitch + 1,), 77, dtype=torch.uint8, device=device)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib().ferry_pack_dispatch(xd.data_ptr(), T, H, seld.data_ptr(), wd.data_ptr(), k, idx.data_ptr(),
                                     ids.data_ptr(), T, k, E, flat[1:].data_ptr(), stream) == 0, last_error()
    assert torch.equal(flat[1:].view(T, pitch).cpu(), want) and int(flat[0]) == 77
    for raw in (payload, flat[1:].view(T, pitch)):
        hx, hw = ops.unpack_dispatch(raw, H, k)
        ux, uw = unpack_dispatch_ref(want, H, k)
        assert torch.equal(hx.cpu(), ux) and torch.equal(hw.cpu().view(torch.int16), uw.view(torch.int16))


@pytest.mark.parametrize('sizes,received,H', [([1], 1, 8), ([5, 0, 3, 7], 6, 64), ([40, 40, 40], 3, 2056),
                                              ([300] * 20, 300, 256), ([16] * 17, 16, 4096)])
@pytest.mark.parametrize('adjacent', [True, False])
def test_reduce_partials_any_rows(device, sizes, received, H, adjacent):
    """Rows in any order, repeated within a group, up to 16 and more entries a row, rows without
    entries, parts and rows that split one tensor and that do not: bit-equal to the fp32 sums in
    group order."""
    from ferry_amd import expert_ops as ops
    rng = np.random.default_rng(sum(sizes) + received)
    rows = [torch.from_numpy(rng.integers(0, received, n)) for n in sizes]
    if len(sizes) == 17:
        rows = [torch.randperm(16) for _ in sizes]     # 17 entries in every row
    g = torch.Generator().manual_seed(H)
    parts = [torch.randn((n, H), generator=g).to(torch.bfloat16) for n in sizes]
    want = reduce_partials_ref(parts, rows, received, H)
    if adjacent:
        dp = torch.cat(parts).to(device).split(sizes)
        dr = torch.cat(rows).to(device).split(sizes)
    else:
        dp, dr = [p.to(device) for p in parts], [r.to(device) for r in rows]
    got = ops.reduce_partials(list(dp), list(dr), received, H, dp[0])
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16))
    for bad in (-1, received):
        r0 = dr[0].clone()
        r0[0] = bad
        with pytest.raises(RuntimeError):
            ops.reduce_partials(list(dp), [r0] + list(dr[1:]), received, H, dp[0])


def test_execute_experts_row_lists(device):
    """Row and column lists that split one tensor and that do not give the same bits, empty groups
    included; int32 lists are taken as before; a list on the host is refused."""
    from ferry_amd import expert_ops as ops
    H, I, T, sizes = 256, 128, 90, [3, 0, 20, 70, 1]
    g = torch.Generator().manual_seed(4)
    cache = (torch.randn((6, 3 * H * I), generator=g) * 0.05).to(torch.bfloat16).to(device)
    x = torch.randn((T, H), generator=g).to(torch.bfloat16).to(device)
    w = torch.rand((T, 2), generator=g).to(torch.bfloat16).to(device)
    rows = torch.randint(T, (sum(sizes),), generator=g).to(device)
    cols = torch.randint(2, (sum(sizes),), generator=g).to(device)
    slots = [5, 1, 0, 2, 3]
    base = ops.execute_experts(cache, x, w, slots, rows.split(sizes), cols.split(sizes), H, I)
    assert [tuple(b.shape) for b in base] == [(n, H) for n in sizes]
    for f in (torch.clone, lambda t: t.to(torch.int32)):
        other = ops.execute_experts(cache, x, w, slots, [f(t) for t in rows.split(sizes)],
                                    [f(t) for t in cols.split(sizes)], H, I)
        assert all(torch.equal(a, b) for a, b in zip(base, other))
    with pytest.raises(RuntimeError):
        ops.execute_experts(cache, x, w, slots, [t.cpu() for t in rows.split(sizes)], cols.split(sizes), H, I)
    with pytest.raises(RuntimeError):
        ops.execute_experts(cache, x, w, [6, 1, 0, 2, 3], rows.split(sizes), cols.split(sizes), H, I)


@pytest.mark.parametrize('counts,entries', [
    ([16, 17, 20, 0, 24], 2048),          # chains of 1, 4 and 8; the longest that 2048 entries allow is 16
    ([32, 33, 15], 2048),                 # 16 and 17 steps
    ([1024, 1025, 1023, 16], 130000),     # the longest listed row
    ([1, 2000], 2001),
])
def test_reduce_rows_of_many_entries(device, counts, entries):
    """Rows of up to and past 16 and 1024 entries among others, in any order, with the workspace that
    holds chains of them and with the smallest: bit-equal to the fp32 sums in order, nothing written
    past the workspace's size."""
    from ferry_amd._lib import last_error, lib
    H = 24
    rng = np.random.default_rng(entries + len(counts))
    rows = len(counts) + -(-(entries - sum(counts)) // 7)
    row_of = np.concatenate([np.repeat(np.arange(len(counts)), counts),
                             len(counts) + np.arange(entries - sum(counts)) // 7])
    row_of = torch.from_numpy(rng.permutation(row_of))
    part = torch.randn((entries, H), generator=torch.Generator().manual_seed(entries)).to(torch.bfloat16)
    want = reduce_partials_ref([part], [row_of], rows, H)
    dp, dr = part.to(device), row_of.to(device)
    small, full = lib().ferry_reduce_rows_workspace_bytes(rows), lib().ferry_reduce_rows_full_workspace_bytes(rows, entries)
    assert small < full
    stream = torch.cuda.current_stream().cuda_stream
    for nbytes in (full, full - 4, small):
        out = torch.full((rows, H), float('nan'), dtype=torch.bfloat16, device=device)
        ws = torch.full((full // 4 + 1,), -5, dtype=torch.int32, device=device)
        assert lib().ferry_reduce_rows(dp.data_ptr(), entries, H, dr.data_ptr(), rows, out.data_ptr(), ws.data_ptr(),
                                       nbytes, stream) == 0, last_error()
        assert torch.equal(out.cpu().view(torch.int16), want.view(torch.int16)), nbytes
        assert int(ws[rows]) == 0 and int(ws[-1]) == -5
        if nbytes != full:
            assert (ws[small // 4:] == -5).all()


def test_more_rows_than_one_grid_holds(device):
    """2^24 packets and received rows (2^32 threads, where a launch's thread count wraps, if each had a
    workgroup of its own): the first, the last and those about the largest grid."""
    from ferry_amd import expert_ops as ops
    n, H, k = 1 << 24, 8, 1
    raw = torch.randint(256, (n, 2 * H + 3 * k), dtype=torch.uint8, device=device)
    x, w = ops.unpack_dispatch(raw, H, k)
    for a in (0, (1 << 22) - 2, n - 4):
        b = slice(a, a + 4)
        assert torch.equal(x[b].view(torch.uint8), raw[b, :2 * H]) and torch.equal(w[b].view(torch.uint8), raw[b, 2 * H:-k])
    del raw, w
    rows = torch.arange(n, device=device)
    out = ops.reduce_partials([x], [rows.flip(0)], n, H, x)
    for a in (0, (1 << 22) - 2, n - 4):
        want = x[n - a - 4:n - a].flip(0)
        assert ((out[a:a + 4] == want) | want.isnan()).all()


def test_device_layout_slot_tables(device):
    """slot_of as an array, list, dict and CUDA tensor leads to the same groups; an active expert
    without a slot is refused."""
    from ferry_amd.layout import device_layout
    E, k, T = 12, 3, 20
    sel, _ = _routing(T, E, k, 6, np.random.default_rng(0))
    active = sorted(set(sel.reshape(-1).tolist()))
    table = np.full(E, -1)
    table[active] = np.arange(len(active))[::-1]
    forms = (table, table.tolist(), {e: table[e] for e in active}, torch.from_numpy(table).to(device))
    for slot_of in forms:
        groups = device_layout(sel.numpy(), None, T, 0, E, slot_of)['groups']
        assert [(g[0], g[3]) for g in groups] == [(e, int(table[e])) for e in active]
    table[active[1]] = -1
    with pytest.raises(AssertionError, match='not cached'):
        device_layout(sel.numpy(), None, T, 0, E, table)
