"""The host tables of the resident 2D time loop (resident.py): every cell has
one owner that marches over it, and what a thread reads and writes stays within
its strip and its border rows."""
import random

import numpy as np
import pytest

from pysit_amd import resident

# rows of a thread's column (plain, PML), threads, jobs of an exchange wave,
# tags of a border: as the library reports them
LIMITS = (9, 5, 512, 6, 64)


def check_strip(plan, d, R):
    nr, nzc, fl, fr = int(d[2]), int(d[21]), int(d[4]), int(d[5])
    items = plan.items[d[28]]
    a = plan.owner_base[d[28]]
    owner = plan.owner[a:a + nr * nzc].reshape(nr, nzc, 2)
    assert (owner >= 0).all()
    cells, exchange = 0, 0
    for w in range(LIMITS[2] // 64):
        wave = items[64 * w:64 * w + 64].astype(np.int64)
        kind = (wave[0, 1] // resident.KIND) & 3
        assert ((wave[:, 1] // resident.KIND & 3) == kind).all()
        if kind == 3:
            exchange += wave[0, 0] < d[23]
            continue
        rows_most = LIMITS[0] if kind == 1 else LIMITS[1]
        first = (wave[0, 2] >> 16) & 0xff
        assert ((wave[:, 2] >> 16 & 0xff) == first).all()
        for t, (base, flags, bits, where) in enumerate(wave):
            col, alias = where & 0xffff, where >> 16
            assert 0 <= alias < LIMITS[2] and items[alias, 3] & 0xffff == col
            step = -1 if flags & resident.REV else 1
            if not bits & 0xffff:  # nothing of its own: the same march as the thread it repeats
                assert items[alias, 2] & 0xffff and (items[alias, :2] & 1).tolist() == [base & 1, flags & 1]
                assert items[alias, 0] == base
            own = [j for j in range(rows_most) if bits >> j & 1]
            late = bits >> 24 & 1
            assert not own or own == list(range(first + late, rows_most))
            assert (fl <= col < nzc - fr) == (kind == 1)
            for j in range(first, rows_most):
                assert 0 <= base + step * j < nr
            # the rows of the stencil around the march
            for j in (first - R, rows_most - 1 + R):
                assert -R <= base + step * j < nr + R
            for j in own:
                assert tuple(owner[base + step * j, col]) == (64 * w + t, j)
                cells += 1
            rows = [base + step * j for j in own]
            if rows:
                top, bot = flags & (2 | 32), flags & (4 | 64)
                assert bool(top) == (min(rows) < R) and bool(bot) == (max(rows) + R >= nr)
                # a march waits at its begin for the border it starts at
                assert not (flags & (4 | 32) if step > 0 else flags & (2 | 64))
    assert cells == nr * nzc and exchange == d[23] >= 1


@pytest.mark.parametrize("seed", range(6))
def test_tables_cover_the_grid_and_stay_in_bounds(seed):
    rng = random.Random(seed)
    held = 0
    for _ in range(12):
        shape = (rng.randint(12, 1200), rng.randint(10, 1500 if seed % 2 else 400))
        pml = tuple(tuple(min(rng.choice([0, rng.randint(1, 25)]), n // 3) for _ in range(2)) for n in shape)
        R, item = rng.randint(1, 4), rng.choice([4, 8])
        keys = ((shape, pml, rng.randint(1, 3)),) * rng.choice([1, 2, 5, 20])
        plan = resident.Plan(keys, R, item, LIMITS, 256)
        if not plan.ok:
            continue
        held += 1
        strips = plan.strips
        assert np.diff(plan.group_begin).max() <= 256
        for si in range(len(keys)):
            mine = strips[strips[:, 0] == si]
            assert mine[0, 1] == 0 and mine[-1, 1] + mine[-1, 2] == shape[0]
            assert (mine[1:, 1] == mine[:-1, 1] + mine[:-1, 2]).all() and (len(mine) == 1 or (mine[:, 2] >= R).all())
            assert (mine[:, 19] == np.append(-1, mine[:-1, 22])).all()
            assert (mine[:, 20] == np.append(mine[1:, 22], -1)).all()
        copies = np.stack(resident.lds_copies(strips, -(-R // (16 // item)), R, strips[:, 2] * keys[0][2]))
        assert resident.lds_offsets(copies, strips[:, 2], item)[-1].max() + 32 <= resident.LDS_BYTES
        _, one = np.unique(strips[:, 28], return_index=True)
        for k in one:
            check_strip(plan, strips[k], R)
    assert held


def test_a_capturing_stream_builds_no_tables(monkeypatch):
    """Under capture a batch without resident tables takes the step kernels
    and builds nothing; outside it asks for them again."""
    import torch
    from pysit_amd import _native, device
    built = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(device.ResidentTables, "build", lambda batch, always: built.append(batch))
    b = object.__new__(device.DeviceBatch)
    b._resident, b._resident_always, b.persistent, b.dtype = None, False, False, np.dtype(np.float64)
    assert b._resident_for(_native.Batch(), 0, 100) is None and b.resident_tables() is None
    assert not built and b._resident is None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert b.resident_tables() is None and built == [b]


def test_kept_plans_drop_one_at_a_time_and_serve_threads():
    """Past its bound a store of plans drops the value used longest ago, not
    all of them, and threads that fill and read it beyond the bound each get
    the value of their key."""
    import threading
    kept = resident._Kept(4)
    made = []
    get = lambda k: kept.get(k, lambda: made.append(k) or ("plan", k))
    for k in (0, 1, 2, 3, 0, 4, 0, 2):  # 1 goes when 4 comes
        assert get(k) == ("plan", k)
    assert made == [0, 1, 2, 3, 4] and len(kept) == 4
    wrong = []

    def work(seed):
        rng = random.Random(seed)
        for _ in range(3000):
            k = rng.randrange(12)
            if get(k) != ("plan", k):
                wrong.append(k)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong and len(kept) == 4


def test_a_survey_of_many_apertures_makes_each_plan_once(monkeypatch):
    made = []
    init = resident.Plan.__init__
    monkeypatch.setattr(resident.Plan, "__init__", lambda self, *a: made.append(a[0]) or init(self, *a))
    resident._PLANS.clear()
    for _ in range(2):
        for w in range(60, 100):
            resident.Plan.of((((w, 60), ((6, 6), (5, 5)), 1),), 2, 4, LIMITS, 256)
    assert len(made) == 40


class _Device(object):
    multi_processor_count = 256


@pytest.mark.parametrize("shape,pml,dtype,held", [((77, 67), 8, np.float32, True), ((116, 288), 50, np.float64, False)])
def test_a_batch_is_built_once_whichever_loop_takes_it(monkeypatch, shape, pml, dtype, held):
    """The route is known from the shots' sizes: neither loop's batch is made
    only to be thrown away, and an entry outside the grid reaches the check
    that refuses it."""
    import types
    import torch
    from pysit_amd import autotune
    from pysit_amd.modeling import temporal_modeling as tmod
    from tests.problems import Synthetic
    made = []

    class Batch(object):
        def __init__(self, *a, **kw):
            made.append("resident")

    monkeypatch.setattr(resident.N, "resident_limits", lambda: LIMITS)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda dev: _Device)
    monkeypatch.setattr(tmod, "DeviceBatch", Batch)
    monkeypatch.setattr(autotune, "tuned_batch", lambda *a, **kw: made.append("steps"))
    mesh = types.SimpleNamespace(dim=2, deltas=(0.01, 0.01))
    solver = types.SimpleNamespace(supports={"equation_dynamics": "time"}, mesh=mesh, dt=1e-3, dtype=dtype,
                                   spatial_accuracy_order=8)
    tools = tmod.TemporalModeling(solver)
    g = Synthetic(shape, ((pml, pml), (pml, pml)), (0.01, 0.01), 20, 8).geometry()
    tools.make_batch([g], None)
    assert made == (["resident"] if held else ["steps"])
    del made[:]
    g.src[0][0] = shape[0], 3
    tools.make_batch([g], None)
    assert made == ["steps"]  # whose batch refuses the entry


class _Loop(object):
    """Resident tables that take ``size`` bytes and ``slot`` bytes of working
    space per slot, 32 slots at least."""

    def __init__(self, size, slot):
        self.size, self.slot_bytes, self.room = size, slot, 0

    def reserve(self, max_nt, room):
        return self.size + self.slot_bytes * max(32, room // self.slot_bytes)

    def held(self):
        return 0


@pytest.mark.parametrize("loop", [0, 1000, 40000, 10 ** 9])
def test_a_memory_budget_counts_the_loop(loop):
    """The schedule leaves room for the loop's buffers; where they would cost
    the kind of the schedule or all of it, the batch does without them, and a
    budget that held a schedule before still does.  What is left over goes to
    the working space, and segments stay as few as the budget holds."""
    import torch
    from pysit_amd import device
    nt, n, nodes = 200, 1000, 30

    def batch(budget, tables):
        b = object.__new__(device.DeviceBatch)
        b._resident, b.schedule, b.memory_budget, b.max_snaps, b.ic_window = tables, "auto", budget, None, 64
        b.dtype, b.dim, b.total_n, b.max_nt, b.dw = np.dtype(np.float32), 2, n, nt, None
        b.adj_inj = (None, None, torch.zeros(nodes + 1))
        return b

    state, ckpt, slot, base = 7 * n * 4, 4 * n * 4, n * 4, 7 * n * 4 + 12 * n
    for budget in range(base + 60000, base + nt * (slot + nodes * 4) + 40000, 7777):
        plain = batch(budget, False)
        try:
            K = plain.plan_segments(True)
        except MemoryError:
            continue
        b = batch(budget, _Loop(loop, 2 * nodes * 4))
        Kb = b.plan_segments(True)
        assert (plain.snaps is None) == (b.snaps is None)
        if b._resident is False:
            assert Kb == K and b.levels == plain.levels
        elif b.snaps is None:
            t = b._resident
            levels = b.levels if Kb < nt else []
            counts = [-(-a // k) for a, k in zip([nt] + levels, levels)]
            need = (levels or [nt])[-1] * slot + sum(counts) * ckpt + (state if levels else 0)
            work = max(t.room, 32 * t.slot_bytes)
            assert t.room >= 0 and base + need + loop + work <= budget
            if len(levels) == 1:  # one segment fewer would not fit
                fewer = counts[0] - 1
                assert fewer == 0 or base + -(-nt // fewer) * slot + fewer * ckpt + state + loop + 32 * t.slot_bytes > budget


def test_a_kept_plan_belongs_to_its_grouping(monkeypatch):
    """Another rule that groups the shots makes its own plan, whatever is kept
    from an earlier one."""
    keys = (((61, 53), ((6, 7), (5, 8)), 1),) * 3
    one = resident.Plan.of(keys, 4, 8, LIMITS, 256)
    rule = resident.plan_groups
    monkeypatch.setattr(resident, "plan_groups", lambda shots, cus: rule(shots, len(shots[0].cut(1e9))))
    other = resident.Plan.of(keys, 4, 8, LIMITS, 256)
    assert len(one.group_begin) == 2 and len(other.group_begin) > 2


def _on_cpu(monkeypatch):
    """Batches whose tables are built in host memory."""
    import torch
    from pysit_amd import device
    monkeypatch.setattr(resident.N, "resident_limits", lambda: LIMITS)
    monkeypatch.setattr(resident.N, "tile_rows", lambda dim, code, axis: (16, 8)[axis] if dim == 3 else 8)
    monkeypatch.setattr(device, "_dev", lambda: torch.device("cpu"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda dev: _Device)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self, *a: self)
    return device.DeviceBatch


def _shared(probs, seed):
    """Geometries of which the odd ones share the first one's receivers, given
    in no order, as a survey's shots share an operator."""
    g = [p.geometry() for p in probs]
    order = np.random.default_rng(seed).permutation(g[0].adj[1].size)
    g[0].adj = tuple(a[order] for a in g[0].adj)
    g[0].rec = tuple(a[order[::-1]] for a in g[0].rec)
    for other in g[1::2]:
        other.adj, other.rec, other.nrec = g[0].adj, g[0].rec, g[0].nrec
    return g


@pytest.mark.parametrize("shape,tiles", [((70, 150), "shot"), ((70, 150), "interleave"), ((20, 30, 140), "shot")])
def test_entry_tables_hold_every_entry_in_its_order(monkeypatch, shape, tiles):
    """The injection and receiver tables against the entries one by one:
    tiles, then nodes, then the entries of a node as given; receivers' entries
    as given; also where shots share their entries."""
    from tests.problems import Synthetic
    make = _on_cpu(monkeypatch)
    dim = len(shape)
    probs = [Synthetic(shape, ((4, 5),) * dim, (0.01,) * dim, 12, 4, seed=i, n_rec=9, n_src=2) for i in range(3)]
    b = make(_shared(probs, 1), probs[0].model, (0.01,) * dim, probs[0].dt, 4, tile_order=tiles)
    lists = {tuple(t[:2]): i for i, t in enumerate(b.tiles.numpy().reshape(-1, 4))}
    for tables, entries in ((b.fwd_inj, [s.src for s in b.shots]), (b.adj_inj, [s.adj for s in b.shots])):
        want = {}
        for si, (pos, chan, w) in enumerate(entries):
            tile, local = b._tile_of_pos(b.shots[si], b.tiles_info[si][0], pos)
            for t, l, c, v in zip(tile, local, chan, w):
                want.setdefault((lists[si, t], int(l)), []).append((si, c, v))
        ptr, node, nptr, chan, w, shot = (t.numpy() for t in tables)
        got = {}
        for t in range(b.n_tiles):
            for n in range(ptr[t], ptr[t + 1]):
                got[t, int(node[n])] = [(shot[n], chan[e], w[e]) for e in range(nptr[n], nptr[n + 1])]
        assert list(got) == sorted(want) and got == want
    recs, at, w = b.recs.numpy().reshape(-1, 4), b.rec_idx.numpy(), b.rec_w.numpy()
    rows = iter(recs)
    for si, s in enumerate(b.shots):
        idx = (s.rec[0] // shape[-1]) * b.zs[si] + s.rec[0] % shape[-1]
        for r in range(s.nrec):
            shot, k, e0, e1 = next(rows)
            mine = s.rec[1] == r
            assert (shot, k) == (si, r) and np.array_equal(at[e0:e1], idx[mine]) and np.array_equal(w[e0:e1], s.rec[2][mine])


@pytest.mark.parametrize("z", [30, 63])
def test_resident_entries_of_shared_operators(monkeypatch, z):
    """The loop's source and receiver tables against the entries one by one,
    where shots share entries and have their nodes in one z tile or in two."""
    import ctypes
    from tests.problems import Synthetic
    make = _on_cpu(monkeypatch)
    probs = [Synthetic((150, 130), ((6, 7), (5, 8)), (0.01, 0.01), 12, 8, seed=i, n_rec=9, rec_z=z) for i in range(3)]
    b = make(_shared(probs, 2), probs[0].model, (0.01, 0.01), probs[0].dt, 8, resident=True)
    assert b.adj_by_node == (z == 30)
    q, R, V, hc = b.resident_tables().struct, 4, 4, 1

    def view(ptr, n, kind=ctypes.c_int):
        return np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(kind)), (n,))

    strips = view(q.strips, 32 * q.n_strips).reshape(-1, 32)
    plan = resident.ResidentTables.plan(b.shots, R, 4, b.dev, True)

    def strip_of(si, node):
        x, zz = divmod(int(node), b.shots[si].shape[1])
        st = [k for k, d in enumerate(strips) if d[0] == si and d[1] <= x < d[1] + d[2]]
        assert len(st) == 1
        return st[0], x - int(strips[st[0]][1]), zz

    for way, entries in enumerate(([s.src for s in b.shots], [s.adj for s in b.shots])):
        n = q.n_inj[way]
        nptr = view(q.inj_nptr[way], n + 1)
        chan, w = view(q.inj_chan[way], nptr[-1]), view(q.inj_w[way], nptr[-1], ctypes.c_double)
        lds, shot = view(q.inj_lds[way], n), view(q.inj_shot[way], n)
        finfo = view(q.finfo[way], 1024 * (1 + strips[:, 29 + way].max())).reshape(-1, 512, 2)
        i = 0
        for si, (pos, c, v) in enumerate(entries):
            flat = pos[:, 0] * 130 + pos[:, 1]
            for node in np.unique(flat):
                mine = flat == node
                assert shot[i] == si and np.array_equal(chan[nptr[i]:nptr[i + 1]], c[mine])
                assert np.array_equal(w[nptr[i]:nptr[i + 1]], v[mine])
                st, row, zz = strip_of(si, node)
                d = strips[st]
                assert d[10 + 2 * way] <= i < d[11 + 2 * way]
                # the thread that owns the cell reads it where the value is put
                t, step = plan.owner[plan.owner_base[d[28]] + row * d[21] + zz // V]
                first, steps = finfo[d[29 + way], t]
                assert steps >> step & 1
                assert lds[i] == (first + bin(steps & ((1 << step) - 1)).count("1")) * V + zz % V
                i += 1
        assert i == n
    lds, at = view(q.rec_lds, q.n_rec_nodes), view(q.rec_node, len(b.rec_w))
    e = 0
    for si, s in enumerate(b.shots):
        for node in s.rec[0][np.argsort(s.rec[1], kind="stable")]:
            st, row, zz = strip_of(si, node)
            d = strips[st]
            assert d[8] <= at[e] < d[9] and lds[at[e]] == ((R + row) * (d[21] + hc) + hc) * 16 + zz * 4
            e += 1
    assert e == len(b.rec_w)


def test_chunks_of_a_long_run_fit_the_grid():
    """A record of few receivers and many steps is cut to chunks that the
    receivers' kernel can number."""
    t = object.__new__(resident.ResidentTables)
    for nodes in (1, 10, 84, 100000):
        t.slot_bytes = nodes * 4
        for nt in (5, 100, 10 ** 6, 10 ** 8):
            for room in (0, 10 ** 6, resident.CHUNK_BYTES, 10 ** 11):
                slots = t.chunk_slots(nt, room)
                assert 1 <= slots <= nt and -(-slots // 8) <= 65535
                assert slots * t.slot_bytes <= max(room, 32 * t.slot_bytes)


def test_buffers_given_back_wait_for_the_stream_that_used_them(monkeypatch):
    """A working space or source buffer dropped by a run on another stream
    than it was allocated on is not given out before that run is done."""
    import torch
    from pysit_amd import device
    used = []

    class Buffer(object):
        def record_stream(self, stream):
            used.append((self, stream))

    monkeypatch.setattr(torch.cuda, "current_stream", lambda: "other")
    t = object.__new__(resident.ResidentTables)
    work = Buffer()
    t._work = 32, work
    t.release()
    assert t._work is None and used == [(work, "other")]
    t.release()
    b = object.__new__(device.DeviceBatch)
    b.release_sources()
    b._inj_pre = Buffer()
    b.release_sources()
    assert b._inj_pre is None and len(used) == 2
