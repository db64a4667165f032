"""Calls whose kernels read inputs from and write results to host memory, at
the sizes where their tiles and launches end: one row, one row either side of
a tile, several launches through the ring's slots, and more launches than
slots; near and wide coordinates (one and two planes of the transfer form);
and at every line of a rule that chooses a form.  Whole numbers, so every
comparison is exact."""
from __future__ import annotations

import ctypes as C
import itertools
import sys
import threading

import numpy as np
import pytest

import _oracle as O
from cudaedgeelimination_amd import _lib, backend
from cudaedgeelimination_amd import workloads as W
from cudaedgeelimination_amd.graph import CEIL_2D, EUC_2D, GraphSnapshot
from cudaedgeelimination_amd.resident import JvFleet, JvSession, KoptBatch, KoptServer

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def graph(seed, n, dtype, box):
    rng = np.random.default_rng(seed)
    return W.knn_graph(rng.integers(0, box, n), rng.integers(0, box, n), dtype, 8)


@pytest.mark.parametrize("box", [1_000_000, 1 << 30])
@pytest.mark.parametrize("k, rows", [(3, 1), (3, 63), (3, 65), (3, 70_000), (4, 15), (4, 17), (4, 2_731),
                                     (5, 1), (5, 3), (5, 5), (5, 315), (5, 316), (5, 4_799), (5, 20_011),
                                     # the whole ring in one launch, and two slots: near, then wide
                                     (5, 4_760), (5, 4_764), (5, 3_848), (5, 3_852)])
def test_rows_match_oracle(ctx, k, rows, box):
    say(f"direct k={k} rows={rows} box={box}")
    dtype = CEIL_2D if rows % 2 else EUC_2D
    g = graph(rows + k, 700, dtype, box)
    tasks = W.kopt_tasks(rows, g, np.full(rows, k, np.uint8))
    table = backend.build_kopt_reconnect_table(k)
    want, _, _ = O.kopt_costs(g.x, g.y, dtype, k, tasks)
    for _ in range(2):  # caches empty, then up to date (the launch before the checks)
        got, _, usage = backend.evaluate_kopt_template_costs_cuda(g, table, tasks, ctx)
        assert np.array_equal(got, want)
    assert usage.snapshot_hit and usage.template_hit and usage.workspace_hit


@pytest.mark.parametrize("rows", [7, 3_000])
def test_checks_beside_the_launch(ctx, rows):
    """A refused row leaves the caller's buffer alone and the next call right;
    coordinates that differ from the cached ones in one late node are seen."""
    say(f"direct checks rows={rows}")
    k = 5
    g = graph(rows, 900, EUC_2D, 1_000_000)
    tasks = W.kopt_tasks(rows, g, np.full(rows, k, np.uint8))
    table = backend.build_kopt_reconnect_table(k)
    want, _, _ = O.kopt_costs(g.x, g.y, EUC_2D, k, tasks)
    got, _, _ = backend.evaluate_kopt_template_costs_cuda(g, table, tasks, ctx)
    assert np.array_equal(got, want)
    for field, value in (((0, 3), 900), ((0, 3), -5), ((0, 1), None), ((2, 2), None)):
        bad = tasks.copy()
        row = bad["port_nodes"][rows - 1]
        if value is not None:
            row[field[1]] = value
        elif field == (0, 1):
            row[1] = row[0]  # a loop
        else:
            row[2], row[3] = row[1], row[0]  # the first deleted edge again
        out = np.full(rows * 208, -7, np.int64)
        status = _lib.lib().ee_kopt_eval_costs(
            ctx.handle, _lib.ptr(g.x), _lib.ptr(g.y), g.dimension, EUC_2D, k, _lib.ptr(table.templates), 208,
            table.generator_hash, _lib.ptr(bad), rows, _lib.ptr(out), None)
        assert status == 1 and (out == -7).all()
        got, _, usage = backend.evaluate_kopt_template_costs_cuda(g, table, tasks, ctx)
        assert np.array_equal(got, want) and usage.snapshot_hit
    moved = g.copy()
    node = int(tasks["port_nodes"][0, 0])
    moved.x[node] += 1000
    got, _, usage = backend.evaluate_kopt_template_costs_cuda(moved, table, tasks, ctx)
    want2, _, _ = O.kopt_costs(moved.x, moved.y, EUC_2D, k, tasks)
    assert not usage.snapshot_hit and np.array_equal(got, want2) and not np.array_equal(want2, want)


def test_wider_tables(ctx):
    """Tables of other sizes than the canonical ones: one template (many
    tiles per launch) and all 945 matchings of ten ports (wide rows)."""
    k = 5
    g = graph(11, 400, EUC_2D, 1 << 30)
    canon = backend.build_kopt_reconnect_table(k)
    tasks = W.kopt_tasks(3, g, np.full(30_000, k, np.uint8))
    want, _, _ = O.kopt_costs(g.x, g.y, EUC_2D, k, tasks)
    one = backend.KOptReconnectTable(k, canon.templates[17:18].copy(), 99)
    got, _, _ = backend.evaluate_kopt_template_costs_cuda(g, one, tasks, ctx)
    assert np.array_equal(got, want.reshape(-1, 208)[:, 17])
    wide = backend.KOptReconnectTable(k, np.tile(canon.templates, 5)[:945].copy(), 98)
    got, _, _ = backend.evaluate_kopt_template_costs_cuda(g, wide, tasks[:2_000], ctx)
    assert np.array_equal(got.reshape(-1, 945), np.tile(want.reshape(-1, 208)[:2_000], 5)[:, :945])


@pytest.mark.parametrize("box", [1_000_000, 1 << 30])
def test_batch_download_ranges(ctx, box):
    """Resident cells read back in ranges that start and end on, before and
    after the transfer kernel's tiles (512 cells) and slots (2^19 near cells,
    419,328 wide ones), at odd offsets, and whole."""
    say(f"batch download box={box}")
    k, rows = 5, 5_300  # 1,102,400 cells: three slots near or wide
    far = graph(5, 300, CEIL_2D, box)
    near = graph(6, 500, EUC_2D, 1_000_000)
    tasks = [W.kopt_tasks(7, far, np.full(rows, k, np.uint8)), W.kopt_tasks(8, near, np.full(40, 3, np.uint8))]
    want, _, _ = O.kopt_costs(far.x, far.y, CEIL_2D, k, tasks[0])
    small, _, _ = O.kopt_costs(near.x, near.y, EUC_2D, 3, tasks[1])
    batch = KoptBatch(ctx)
    a, b = batch.add_instance(far), batch.add_instance(near)
    batch.set_work([(a, k, rows), (b, 3, 40)], np.concatenate(tasks))
    batch.run()
    assert np.array_equal(batch.segment_costs(1), small)
    slot = 1 << 19 if box == 1_000_000 else 419_328
    for first, count in ((0, len(want)), (0, 1), (1, 511), (3, 512), (511, 513), (7, 65_536), (0, slot),
                         (5, slot + 1), (1, 2 * slot - 1), (9, 2 * slot + 3), (len(want) - 1, 1), (4, 0)):
        assert np.array_equal(batch.download(first, count), want[first:first + count]), (first, count)
    batch.close()


@pytest.mark.parametrize("box", [1_000_000, 1 << 30])
@pytest.mark.parametrize("output", ["costs", "masks"])
@pytest.mark.parametrize("k, rows", [(3, 1), (3, 31), (3, 1_225), (4, 7), (4, 9), (4, 18_424), (5, 1), (5, 9),
                                     (5, 255), (5, 257), (5, 14_001), (5, 44_000)])
def test_made_rows_match_oracle(ctx, k, rows, output, box):
    """Rows made by the wavefronts that evaluate them, at the edges of tiles,
    of the host's groups of 256 rows, and of launches (several slots)."""
    if output == "costs" and rows > 14_001:
        rows = 9_400  # three launches of cells
    say(f"made rows k={k} rows={rows} {output} box={box}")
    g = graph(rows + k, 900, CEIL_2D if rows % 2 else EUC_2D, box)
    tour = W.tour_context(rows, g, 120, 51)
    table = backend.build_kopt_reconnect_table(k)
    first = backend.kopt_cursor_count(tour, k) - rows if rows < 1_000 else 0
    want, positions = O.cursor_tasks(tour.tour, tour.edge_costs, tour.selectable, k, first, rows)
    cells, _, _ = O.kopt_costs(g.x, g.y, g.distance_type, k, want)
    for _ in range(2):  # caches empty, then up to date
        block = backend.evaluate_kopt_cursor_cuda(g, table, tour, k, first, rows, output, ctx)
        assert np.array_equal(block.tasks["port_nodes"], want["port_nodes"])
        assert np.array_equal(block.tasks["deleted_cost"], want["deleted_cost"])
        assert np.array_equal(block.positions, positions)
        if output == "costs":
            assert np.array_equal(block.costs, cells)
        else:
            bits = np.unpackbits(block.masks.view(np.uint8), axis=1, bitorder="little")
            improving = cells.reshape(rows, -1) < want["deleted_cost"][:, None]
            assert np.array_equal(bits[:, :improving.shape[1]].astype(bool), improving)
            assert not bits[:, improving.shape[1]:].any()


@pytest.mark.parametrize("wanted", ["neither", "tasks", "positions"])
@pytest.mark.parametrize("k, rows, output", [(4, 1, "masks"), (5, 9, "masks"), (5, 30_000, "masks"), (3, 65, "costs"),
                                             (5, 4_999, "costs"), (5, 12_001, "costs")])
def test_made_rows_left_out(ctx, k, rows, output, wanted):
    """Made rows and positions reach host memory only where the caller passes
    a buffer; the slots then hold more rows, and the results are the same."""
    say(f"made rows k={k} rows={rows} {output}, wanted: {wanted}")
    g = graph(rows, 900, EUC_2D, 1 << 30 if rows == 4_999 else 1_000_000)
    tour = W.tour_context(rows, g, 200, 75)
    table = backend.build_kopt_reconnect_table(k)
    whole = backend.evaluate_kopt_cursor_cuda(g, table, tour, k, 3, rows, output, ctx)
    rows = len(whole.tasks)
    T = len(table.templates)
    view, produced = tour.view(), C.c_uint32()
    out = {"tasks": np.empty(rows, whole.tasks.dtype), "positions": np.empty((rows, k), np.uint32),
           "costs": np.empty(rows * T, np.int64), "masks": np.empty((rows, (T + 31) // 32), np.uint32)}
    for array in out.values():
        array.view(np.uint8)[...] = 0xA5
    _lib.check(_lib.lib().ee_kopt_cursor_eval(
        ctx.handle, _lib.ptr(g.x), _lib.ptr(g.y), g.dimension, g.distance_type, C.byref(view), k,
        _lib.ptr(table.templates), T, table.generator_hash, 3, rows,
        *(_lib.ptr(out[name]) if name in (wanted, output) else None
          for name in ("tasks", "positions", "costs", "masks")), C.byref(produced), None))
    assert produced.value == rows
    for name, array in out.items():
        if name in (wanted, output):
            assert np.array_equal(array, getattr(whole, name))
        else:
            assert (array.view(np.uint8) == 0xA5).all()


def star(n, hub_degree, seed=3):
    """A k-NN graph with one hub joined to `hub_degree` further nodes."""
    g = graph(seed, n, EUC_2D, 1_000_000)
    have = set(zip(g.edge_u.tolist(), g.edge_v.tolist()))
    extra = [(0, v) for v in range(1, n) if (0, v) not in have][:hub_degree]
    u = np.concatenate([g.edge_u, [e[0] for e in extra]]).astype(np.int32)
    v = np.concatenate([g.edge_v, [e[1] for e in extra]]).astype(np.int32)
    order = np.lexsort((v, u))
    return type(g).from_edges(g.x, g.y, EUC_2D, u[order], v[order])


@pytest.mark.parametrize("degree", [55, 90, 500, 700])
def test_hamilton_verdicts(ctx, degree):
    """Hub rows below and above the 64 neighbours cached in LDS and the 512
    that take verdict bits; replies copied in ranges that cut the groups of
    256 centers; a refused call leaves the last call's replies."""
    say(f"ht verdicts hub degree {degree}")
    g = star(800, degree)
    backend.clear_ht_reply_cuda_cache(ctx)
    e = len(g.edge_u) // 2
    target = (int(g.edge_u[e]), int(g.edge_v[e]))
    centers = np.setdiff1d(np.arange(g.dimension, dtype=np.int32), np.array(target, np.int32))
    deg = np.diff(g.row_offsets).astype(np.int64)[centers]
    woff, wrep = O.ht_hamilton_replies(O.OGraph.from_snapshot(g), target, centers,
                                       int((deg * (deg - 1) // 2).sum()))
    for _ in range(2):
        off, rep, _ = backend.evaluate_ht_hamilton_replies_cuda(g, target, centers, ctx)
        assert np.array_equal(off, woff) and np.array_equal(rep, wrep)
    total = len(wrep)
    for first, count in ((0, 1), (1, 7), (total // 3, total // 2), (total - 1, 1), (5, 0)):
        part = np.full((count, 3), -1, np.int32)
        _lib.check(_lib.lib().ee_ht_copy_replies(ctx.handle, first, count, _lib.ptr(part) if count else None))
        assert np.array_equal(part, wrep[first:first + count])
    with pytest.raises(_lib.InvalidArgument):
        backend.evaluate_ht_hamilton_replies_cuda(g, target, np.array([0, target[1]], np.int32), ctx)
    with pytest.raises(_lib.InvalidArgument):
        backend.evaluate_ht_hamilton_replies_cuda(g, target, np.array([0, g.dimension], np.int32), ctx)
    part = np.empty((total, 3), np.int32)
    _lib.check(_lib.lib().ee_ht_copy_replies(ctx.handle, 0, total, _lib.ptr(part)))
    assert np.array_equal(part, wrep)
    # the same sizes with one node moved: not the resident snapshot
    moved = g.copy()
    moved.x[g.dimension - 1] += 5000
    moved = type(g).from_edges(moved.x, moved.y, EUC_2D, moved.edge_u, moved.edge_v)
    off, rep, usage = backend.evaluate_ht_hamilton_replies_cuda(moved, target, centers, ctx)
    woff, wrep = O.ht_hamilton_replies(O.OGraph.from_snapshot(moved), target, centers,
                                       int((deg * (deg - 1) // 2).sum()))
    assert not usage.graph_hit and np.array_equal(off, woff) and np.array_equal(rep, wrep)


def edges_graph(pairs, n, dtype=EUC_2D, box=1_000_000, seed=5):
    """A snapshot on random points with exactly these edges."""
    rng = np.random.default_rng(seed)
    u, v = (np.array(c, np.int32) for c in zip(*sorted(set(map(tuple, map(sorted, pairs))))))
    return GraphSnapshot.from_edges(rng.integers(0, box, n), rng.integers(0, box, n), dtype, u, v)


def hamilton_oracle(g, target, centers):
    deg = np.diff(g.row_offsets).astype(np.int64)[centers]
    return O.ht_hamilton_replies(O.OGraph.from_snapshot(g), target, centers, int((deg * (deg - 1) // 2).sum()))


@pytest.mark.parametrize("form", ["near", "wide", "ceil"])
@pytest.mark.parametrize("degree", [0, 1, 15, 16, 17, 22, 23, 24, 63, 64, 65, 91, 92])
def test_hamilton_rows_either_side(ctx, degree, form):
    """Complete graphs (rows of one length) around every line of the verdict
    form: 16 neighbours gathered together, one stride for all up to 23, 64
    cached in LDS, 64 words a center on average (92 neighbours take three
    passes); near, 64-bit and CEIL_2D distances; beside them centers without
    edges, in lists that end inside a wavefront."""
    say(f"ht rows degree {degree} {form}")
    n = max(degree + 1, 2)
    pairs = list(itertools.combinations(range(n), 2)) + [(n, n + 1)]  # the target apart
    g = edges_graph(pairs if degree else [(n, n + 1)], n + 7, CEIL_2D if form == "ceil" else EUC_2D,
                    1 << 30 if form == "wide" else 1_000_000, degree + 1)
    alone = np.arange(n + 2, n + 7, dtype=np.int32)  # no edges
    for target in ((n, n + 1), (0, 1)) if degree else ((n, n + 1),):
        rest = np.setdiff1d(np.arange(n + 2, dtype=np.int32), np.array(target, np.int32))
        lists = [rest, np.concatenate([alone[:2], rest, alone[2:3], rest[:3]]), np.tile(rest, 3)[:-1]]
        for centers in lists + ([alone] if degree < 24 else []):
            want = hamilton_oracle(g, target, centers)
            for _ in range(2):
                off, rep, _ = backend.evaluate_ht_hamilton_replies_cuda(g, target, centers, ctx)
                assert np.array_equal(off, want[0]) and np.array_equal(rep, want[1])


@pytest.mark.parametrize("hub", [30, 512, 513])
def test_hamilton_hub_costs_its_own_words(hub):
    """A hub among short rows: what the context keeps follows the centers'
    own rows (all 2,044 words of a row of 512 for each of 3,000 centers would
    be 49 MB, twice), whether the hub is a center, several times, or not."""
    say(f"ht hub {hub}")
    n = 3_000
    g = edges_graph([(i, i + 1) for i in range(1, n - 1)] + [(0, 5 * i + 1) for i in range(hub)], n)
    own = backend.Context(0)
    target = (n - 2, n - 1)
    plain = np.arange(1, n - 2, dtype=np.int32)
    for centers, hubs in ((plain, 0), (np.concatenate([plain[:1_001], [0], plain[1_001:]]).astype(np.int32), 1),
                          (np.tile(np.concatenate([[0], plain[:40]]), 31).astype(np.int32), 31)):
        want = hamilton_oracle(g, target, centers)
        for _ in range(2):
            off, rep, usage = backend.evaluate_ht_hamilton_replies_cuda(g, target, centers, own)
            assert np.array_equal(off, want[0]) and np.array_equal(rep, want[1])
        # the snapshot; centers, counts, bits and offsets, twice and grown at
        # most twofold; or the replies, their counts and offsets
        pairs = hubs * hub * (hub - 1) // 2 + 2 * len(centers)
        words = pairs // 64 + 2 * len(centers)
        assert usage.resident_bytes < 200_000 + 4 * (8 * words + 9 * len(centers)) + (24 * pairs if hub > 512 else 0)
    own.close()


@pytest.mark.parametrize("form", ["near", "wide", "ceil"])
def test_hamilton_three_passes(ctx, form):
    """The count, scan and write passes over more centers than one scan chunk
    holds (1,024), repeated ones among them: a hub beyond 512 neighbours sends
    the call there; 64-bit and CEIL_2D distances, rows beyond the LDS cache."""
    say(f"ht three passes {form}")
    n = 700
    pairs = [(0, i) for i in range(1, 600)] + list(itertools.combinations(range(1, 80), 2))
    pairs += [(i, i + 1) for i in range(1, n - 1)] + [(i, i + 7) for i in range(80, n - 7, 2)]
    g = edges_graph(pairs, n, CEIL_2D if form == "ceil" else EUC_2D, 1 << 30 if form == "wide" else 1_000_000)
    rest = np.arange(1, n, dtype=np.int32)
    for target, centers in (((n - 2, n - 1), np.concatenate([rest[:-2], [0], np.tile(rest[::-1][2:], 3)])),
                            ((1, 2), np.concatenate([np.tile(rest[2:], 2), [0, 0], rest[5:40]]))):
        centers = np.ascontiguousarray(centers, np.int32)
        want = hamilton_oracle(g, target, centers)
        for _ in range(2):
            off, rep, usage = backend.evaluate_ht_hamilton_replies_cuda(g, target, centers, ctx)
            assert np.array_equal(off, want[0]) and np.array_equal(rep, want[1])
        assert usage.resident_bytes > 12 * len(rep) and len(centers) > 1_024
        total = len(rep)
        part = np.empty((total // 2, 3), np.int32)
        _lib.check(_lib.lib().ee_ht_copy_replies(ctx.handle, total // 3, total // 2, _lib.ptr(part)))
        assert np.array_equal(part, rep[total // 3:total // 3 + total // 2])


@pytest.mark.parametrize("hub, centers, takes", [(2, 1 << 22, True), (2, (1 << 22) + 1, False),
                                                 (22, 1 << 20, True), (22, (1 << 20) + 1, False)])
def test_hamilton_bits_limit(hub, centers, takes):
    """32 MiB of verdict bits, at one word and at four words a center, and one
    center more: both forms give the oracle's replies."""
    say(f"ht bits limit hub {hub} centers {centers}")
    n = 1_000
    g = edges_graph([(i, i + 1) for i in range(1, n - 1)] + [(0, 40 * i + 1) for i in range(hub)], n)
    target, base = (n - 2, n - 1), np.arange(2, n - 3, dtype=np.int32)
    off, rep = hamilton_oracle(g, target, base)
    times, left = divmod(centers, len(base))
    own = backend.Context(0)
    got_off, got, usage = backend.evaluate_ht_hamilton_replies_cuda(g, target, np.resize(base, centers), own)
    assert np.array_equal(got, np.concatenate([np.tile(rep, (times, 1)), rep[:off[left]]]))
    per = np.diff(off)
    assert np.array_equal(np.diff(got_off), np.resize(per, centers)) and got_off[0] == 0
    # bits, centers and counts, twice; or centers, counts and offsets (20
    # bytes a center) and the replies
    assert (usage.resident_bytes >= 2 * ((32 << 20) + 8 * centers)) == takes
    own.close()


@pytest.mark.parametrize("rows", [1, 255, 257, 43_520, 43_521, 90_001])
def test_set_work_rows(ctx, rows):
    """Rows checked by the device on their way in, at the edges of its groups
    (256 rows) and slots (43,520): good rows give the oracle's masks, one bad
    row anywhere is refused with the host's message and the batch keeps its
    work."""
    say(f"set_work rows={rows}")
    a, b = graph(21, 400, EUC_2D, 1_000_000), graph(22, 300, CEIL_2D, 1 << 30)
    k3 = rows // 2
    tasks = np.concatenate([W.kopt_tasks(1, a, np.full(k3, 3, np.uint8)),
                            W.kopt_tasks(2, b, np.full(rows - k3, 4, np.uint8))])
    batch = KoptBatch(ctx)
    ia, ib = batch.add_instance(a), batch.add_instance(b)
    batch.set_output("masks")
    segments = [(ia, 3, k3), (ib, 5, 0), (ib, 4, rows - k3)]
    want = []
    for g, k, part in ((a, 3, tasks[:k3]), (b, 4, tasks[k3:])):
        cells, _, _ = O.kopt_costs(g.x, g.y, g.distance_type, k, part)
        bits = cells.reshape(len(part), 4 if k == 3 else 25) < part["deleted_cost"][:, None]
        want.append((bits << np.arange(bits.shape[1])).sum(axis=1).astype(np.uint32))
    want = np.concatenate(want)
    for at in sorted({0, k3 - 1, k3, rows - 1} & set(range(rows))):
        batch.set_work(segments, tasks)
        n = a.dimension if at < k3 else b.dimension
        for port, value, cost in ((2, n, 0), (5, -1, 0), (4, None, 0), (0, None, -1)):
            bad = tasks.copy()
            if cost:
                bad["deleted_cost"][at] = -5
            elif value is None:
                bad["port_nodes"][at, 4:6] = bad["port_nodes"][at, 1::-1]  # the first deleted edge again
            else:
                bad["port_nodes"][at, port] = value
            with pytest.raises(_lib.InvalidArgument, match="negative deleted_cost" if cost else "deleted edge"):
                batch.set_work(segments, bad)
        batch.run()
        assert np.array_equal(batch.download_masks()[:, 0], want)
    batch.close()


@pytest.mark.parametrize("output", ["costs", "masks"])
def test_set_work_without_room(ctx, output):
    """Rows that fit the device with cells that do not (as many as would fill
    it whole): the call fails and the batch has no work, neither the old one's
    tiles with the new rows nor a freed pool; the next work runs."""
    say(f"set_work without room, {output}")
    free, total = C.c_size_t(), C.c_size_t()
    assert _lib.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    count = total.value // (208 * 8) + 1
    g = graph(23, 400, EUC_2D, 1_000_000)
    tasks = W.kopt_tasks(3, g, np.full(500, 5, np.uint8))
    want, _, _ = O.kopt_costs(g.x, g.y, EUC_2D, 5, tasks)
    batch = KoptBatch(ctx)
    instance = batch.add_instance(g)
    batch.set_output(output)
    batch.set_work([(instance, 5, 500)], tasks)
    batch.run()
    rows = np.empty(count, tasks.dtype)
    rows[:] = tasks[7]
    with pytest.raises(_lib.EeError, match="hipMalloc"):
        batch.set_work([(instance, 5, count)], rows)
    del rows
    assert batch.run(3) == 0.0
    if output == "costs":
        with pytest.raises(_lib.InvalidArgument):
            batch.download(0, 1)
    else:
        with pytest.raises(_lib.InvalidArgument):
            batch.download_masks(0, 1)
    batch.set_work([(instance, 5, 500)], tasks)
    batch.set_output("costs")
    batch.run()
    assert np.array_equal(batch.segment_costs(0), want)
    batch.close()


def test_tunings_of_an_older_kernel_are_retuned(ctx, tmp_path):
    """A stored tuning is taken under its own key, and not where its key names
    the kernel's revision 8, before it wrote packed cells and made rows."""
    say("stored tunings")
    g = graph(29, 300, EUC_2D, 1_000_000)
    tasks = W.kopt_tasks(3, g, np.full(64, 4, np.uint8))
    batch = KoptBatch(ctx)
    batch.set_work([(batch.add_instance(g), 4, 64)], tasks)
    cache = tmp_path / "tunings"
    batch.autotune(1, str(cache))
    key = cache.read_text().split()[0]
    assert key.startswith("kopt") and int(key[4:].split("/")[0]) > 8
    planted = "17 13 11 3 192 0"  # options the search never tries
    cache.write_text(f"{key} {planted}\n")
    assert batch.autotune(1, str(cache))["grid"] == 3
    cache.write_text(f"kopt8/{key.split('/', 1)[1]} {planted}\n")
    assert batch.autotune(1, str(cache))["grid"] != 3
    batch.run()
    want, _, _ = O.kopt_costs(g.x, g.y, EUC_2D, 4, tasks)
    assert np.array_equal(batch.segment_costs(0), want)
    batch.close()


@pytest.mark.parametrize("n, neighbors", [(4, 3), (41, 6), (700, 10), (60_000, 8)])
def test_jv_call_inputs(ctx, n, neighbors):
    """The dynamic arrays on their way in (one slot and several; odd counts;
    inactive edges), refused ids, and a snapshot that differs from the resident
    one in one late weight or coordinate."""
    say(f"jv call n={n}")
    rng = np.random.default_rng(n)
    g = W.knn_graph(rng.integers(0, 1_000_000, n), rng.integers(0, 1_000_000, n), EUC_2D, neighbors)
    backend.clear_jv_cuda_cache(ctx)
    for drop in (0, 1, 1 + g.edge_count // 7):
        g.edge_active[rng.permutation(g.edge_count)[:drop]] = 0
        g.rebuild_csr()
        want = O.OGraph.from_snapshot(g).witnesses()
        got, usage = backend.find_jv_witnesses(g, ctx)
        assert np.array_equal(got, want) and usage.static_hit == (drop != 0)
    a = g.adjacency_count
    for name, value, text in (("neighbors", n, "neighbour"), ("neighbors", -1, "neighbour"),
                              ("csr_edge_ids", g.edge_count, "edge id"), ("row_offsets", -2, "non-decreasing")):
        bad = g.copy()
        getattr(bad, name)[(a if name != "row_offsets" else n) - 1] = value
        with pytest.raises(_lib.InvalidArgument, match=text):
            backend.find_jv_witnesses(bad, ctx)
    got, usage = backend.find_jv_witnesses(g, ctx)
    assert np.array_equal(got, want) and usage.static_hit and usage.workspace_hit
    moved = g.copy()
    moved.x[n - 1] += 3000
    moved = type(g).from_edges(moved.x, moved.y, EUC_2D, g.edge_u, g.edge_v, None, g.edge_active)
    got, usage = backend.find_jv_witnesses(moved, ctx)
    assert np.array_equal(got, O.OGraph.from_snapshot(moved).witnesses())
    assert not usage.static_hit and usage.workspace_hit


def test_jv_phase_times(ctx):
    """A call's kernel time holds its kernel: on a complete graph (28,680
    slots that each score 478 neighbours) it is most of the call, and the 0.1
    MB of witnesses after it the smaller part."""
    say("jv phase times")
    g = edges_graph(itertools.combinations(range(240), 2), 240)
    for _ in range(3):
        got, usage = backend.find_jv_witnesses(g, ctx)
    assert np.array_equal(got, O.OGraph.from_snapshot(g).witnesses())
    assert usage.static_hit and usage.kernel_ms > 2 * usage.d2h_ms > 0


@pytest.mark.parametrize("n, neighbors", [(3, 2), (682, 3), (1_023, 3), (1_024, 4), (1_025, 4), (2_049, 5),
                                          (8_193, 6), (50_001, 8)])
def test_session_snapshot_upload(ctx, n, neighbors):
    """Sessions and fleets put their arrays in place in parts of at most 8 KiB: at
    the edges of a part and over several slots, the device's snapshot is the
    graph's, and the hashes (which read the endpoints, weights and flags) and
    witnesses are the host's and the oracle's."""
    say(f"session upload n={n}")
    rng = np.random.default_rng(n)
    graphs = []
    for part in (n, 5, n // 2 + 3):
        g = W.knn_graph(rng.integers(0, 1_000_000, part), rng.integers(0, 1_000_000, part), EUC_2D,
                        min(neighbors, part - 1))
        active = g.edge_active.copy()
        active[:: 7] = 0
        graphs.append(GraphSnapshot.from_edges(g.x, g.y, EUC_2D, g.edge_u, g.edge_v, g.edge_weight, active))
    singles = []
    for g in graphs:
        s = JvSession(ctx, g)
        run = s.run(1)
        assert run.initial_hash == g.content_hash()
        got = s.device_snapshot()
        for name in ("edge_active", "row_offsets", "neighbors", "csr_edge_ids"):
            assert np.array_equal(got[name], getattr(g, name)), name
        s.close()
        s = JvSession(ctx, g)
        singles.append(O.canonical_proof(s.run(100).proof))
        s.close()
    for use_graph in (False, True):
        f = JvFleet(ctx, graphs)
        f.run(100, use_graph)
        for i, proof in enumerate(singles):
            assert O.canonical_proof(f.proof(i)) == proof, i
        f.close()


@pytest.mark.parametrize("order", [(40, 3_000, 40, 900, 3_000), (3_000, 2_900, 1_500, 3_000, 5)])
def test_sessions_one_after_the_other(ctx, order):
    """A context keeps the memory of closed sessions and fleets for the next:
    whatever it held, and whatever is open beside it, the next run's proof is
    a fresh context's."""
    say(f"reused memory {order}")
    graphs = [W.knn_graph(*np.random.default_rng(n).integers(0, 1_000_000, (2, n)), EUC_2D, 4) for n in order]

    def alone(g):
        own = backend.Context(0)
        s = JvSession(own, g)
        proof = O.canonical_proof(s.run(100).proof)
        s.close()
        own.close()
        return proof

    want = [alone(g) for g in graphs]
    beside = JvSession(ctx, graphs[0])
    for _ in range(2):
        for g, proof in zip(graphs, want):
            s = JvSession(ctx, g)
            assert O.canonical_proof(s.run(100).proof) == proof
            s.close()
        f = JvFleet(ctx, graphs)
        f.run(100)
        assert [O.canonical_proof(f.proof(i)) for i in range(len(order))] == want
        f.close()
    assert O.canonical_proof(beside.run(100).proof) == want[0]
    beside.close()


@pytest.mark.parametrize("batching", [True, False])
@pytest.mark.parametrize("rows, slots", [(1, 1), (9, 2), (300, 255), (6_000, 4_097)])
def test_server_in_place(ctx, rows, slots, batching):
    """Served batches read rows, tiles and edge lists from page-locked memory
    and leave cells and witnesses there: near and wide instances in one batch
    (with and without high bytes), several k, a request beyond the batch
    limit, and JV rechecks beside them."""
    say(f"server rows={rows} slots={slots} batching={batching}")
    graphs = [graph(5, 400, EUC_2D, 1_000_000), graph(6, 700, CEIL_2D, 1 << 30)]
    server = KoptServer(ctx, max_batch_cells=20_000, batching=batching)
    ids = [server.add_graph(g) for g in graphs]
    gj = W.knn_graph(*np.random.default_rng(9).integers(0, 1_000_000, (2, 1_000)), EUC_2D, 8)
    jid = server.add_jv_graph(gj)
    edges = np.arange(slots, dtype=np.int32)[::-1] % gj.edge_count
    whole, _ = backend.find_jv_witnesses(gj, ctx)
    requests, want = [], []
    for i, g in enumerate(graphs):
        for k in (3, 4, 5):
            count = rows if k == 5 and i == 1 else min(rows, 40)
            tasks = W.kopt_tasks(rows + k, g, np.full(count, k, np.uint8))
            requests.append((ids[i], k, tasks))
            want.append(O.kopt_costs(g.x, g.y, g.distance_type, k, tasks)[0])
        requests.append((jid, 0, edges))
        want.append(whole[edges])
    for _ in range(3):
        for (got, _), exact in zip(server.wait_many(server.submit_many(requests), 60_000), want):
            assert np.array_equal(got, exact)
    server.close()


def test_two_contexts_on_two_threads():
    """Contexts used side by side, each by its own thread: one reads large
    results (the process's host threads take its tiles), the other runs JV
    calls, sessions and small leaf blocks, whose host phases want those threads."""
    say("two contexts on two threads")
    g = W.knn_graph(*np.random.default_rng(31).integers(0, 1_000_000, (2, 3_000)), EUC_2D, 8)
    rows = W.kopt_tasks(5, g, np.full(6_000, 5, np.uint8))
    table = backend.build_kopt_reconnect_table(5)
    cells, _, _ = O.kopt_costs(g.x, g.y, EUC_2D, 5, rows)
    witnesses = O.OGraph.from_snapshot(g).witnesses()
    own = backend.Context(0)
    s = JvSession(own, g)
    proof = O.canonical_proof(s.run(100).proof)
    s.close()
    own.close()
    wrong, done = [], threading.Event()

    def large():
        try:
            mine = backend.Context(0)
            batch = KoptBatch(mine)
            batch.set_work([(batch.add_instance(g), 5, len(rows))], rows)
            while not done.is_set():
                batch.run()
                if not np.array_equal(batch.segment_costs(0), cells):
                    wrong.append("batch")
            batch.close()
            mine.close()
        except Exception as error:  # noqa: BLE001 - reported by the test
            wrong.append(error)

    thread = threading.Thread(target=large)
    thread.start()
    mine = backend.Context(0)
    for i in range(15):
        got, _, _ = backend.evaluate_kopt_template_costs_cuda(g, table, rows[:100 + 50 * i], mine)
        if not np.array_equal(got, cells[:len(got)]):
            wrong.append("leaf")
        if not np.array_equal(backend.find_jv_witnesses(g, mine)[0], witnesses):
            wrong.append("jv")
        s = JvSession(mine, g)
        if O.canonical_proof(s.run(100).proof) != proof:
            wrong.append("session")
        s.close()
    done.set()
    thread.join()
    mine.close()
    assert not wrong
