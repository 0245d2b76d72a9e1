"""Host tables of the 2D time loop that keeps the wavefield on the chip
(``pysit_amd_resident_run``, csrc/resident2d.hip).

A shot is cut along x into strips of whole rows, one workgroup each; a
workgroup's threads own 16-byte cell columns (4 FP32 or 2 FP64 nodes along z)
over a few rows.  Cells away from the PML and the grid's edges take the plain
update (their waves are *plain*), the others the PML update (*full*).  Shots
that do not fit the GPU together run one group after the other.

Everything here is numpy on the host; :class:`ResidentTables` uploads the
result once per batch geometry.
"""
import collections
import ctypes
import threading
import weakref

import numpy as np

from . import _native as N

# LDS a workgroup may use
LDS_BYTES = 160 * 1024
STRIP_INTS = 32
REV, BEGIN_TOP, BEGIN_BOT, KIND, END_TOP, END_BOT = 1, 2, 4, 8, 32, 64
XTYPE, PXTOP, PXBOT = 1, 2, 4
# cost model of a step, in plain rows of a thread (about 600 cycles): a PML
# row, the exchange wave's own work and the factor of the work beside it (a
# border that is late holds up the neighbours too), what a step spends around
# its rows, and the part of the workgroup's whole work that adds to its longest
# SIMD's.  Fitted to the step times of 11 batches: 77 x 67 to 1041 x 341, FP32
# and FP64, 1 to 32 shots; models with the wait for a neighbour as a cost of
# its own chose fewer, higher strips for few shots, up to 1.5 times slower.
FULL_COST = 6.0
EXCHANGE_COST = 1.5
EXCHANGE_SHARE = 1.5
STEP_COST = 2.0
SHARE_COST = 1.0
# what a step of the step kernels costs, in the same unit: launch and latency,
# and the bytes of one field that add 1
STEP_KERNEL_COST = 35.0
STEP_KERNEL_BYTES = 30000.0
# device memory for the source values and receiver nodes of a chunk of slots
# where no memory budget is set, and the slots a chunk has at least: each chunk
# is a launch, which loads and stores the state (55 us for 1 shot of
# 1041 x 341 nodes or 4 of 541 x 241, 100 us for 16 of 1041 x 341; a step takes
# 6, 7 and 18 us)
CHUNK_BYTES = 256 << 20
CHUNK_LEAST = 32
# slots of a chunk at most: the receivers' kernel takes 8 slots a workgroup
# along its grid's second axis, which has 65535 at most
CHUNK_SLOTS = 8 * 65535
# shorter runs than this many slots go through the step kernels: a resident
# launch loads and stores the whole state
RESIDENT_MIN_SLOTS = 8
# polls of about 1 us (16 s) before a wait for a neighbour gives up: a strip
# may start late where another stream's kernels hold compute units
SPIN = 1 << 24


class _Words(object):
    """Pinned host words that a device can write, one per user: the word of
    an expired wait belongs to one batch.  A freed word is the last to be
    given out again: a launch of a batch that is gone may still write it."""

    BLOCK = 1024

    def __init__(self):
        self._lock = threading.Lock()
        self._free = collections.deque()

    def take(self, owner):
        """A word (a view of one int32) that is ``owner``'s while it lives."""
        import torch
        with self._lock:
            if not self._free:
                block = torch.zeros(self.BLOCK, dtype=torch.int32).pin_memory()
                self._free.extend(block[i:i + 1] for i in range(self.BLOCK))
            word = self._free.popleft()
        word[0] = 0
        weakref.finalize(owner, self._free.append, word)
        return word


_WORDS = _Words()


def z_columns(nz, nzl, nzr, R, V):
    """(cells of a row, full cells at the left, full cells at the right): a
    cell is full if a node within R of it is a PML node, an edge node or
    beyond the grid."""
    nzc = -(-nz // V)
    fl = min(nzc, -(-(max(nzl, 1) + R) // V))
    # the first cell whose last node reaches the right band
    first = max(0, -(-(nz - max(nzr, 1) - R - (V - 1)) // V))
    fr = max(0, nzc - first)
    if fl + fr >= nzc:
        return nzc, nzc, 0
    return nzc, fl, fr


def _groups(nr, n):
    """n row groups (first row, rows) of nr rows, the larger ones first."""
    base, extra = divmod(nr, n)
    out, r = [], 0
    for g in range(n):
        k = base + (g < extra)
        out.append((r, k))
        r += k
    return out


class Layout(object):
    """How the threads of one workgroup share a strip of ``nr`` rows with
    ``plain`` and ``full`` cell columns.  The threads of a kind take row
    groups column by column, the groups at the strip's borders first: a wave
    with one of them waits for the neighbours' rows.  PML rows near a border
    may be groups of one row, so that little is left to do after the wait.
    ``waves``: per wave its kind (1 plain, 2 full, 3 exchange, 0 idle) and its
    first thread among those of its kind; ``cost``: a step in plain rows."""

    def __init__(self, nr, plain, full, limits, border, R, alone):
        self.nr, self.plain, self.full = nr, plain, full
        rp, rf, threads, jobs, tags = limits
        R = 0 if alone else R  # no neighbour's rows to wait for
        n_waves = threads // 64
        best = None
        plains = [(pg, self._kind_waves(1, pg, plain, 1.0, nr, R)) for pg in self._plain_groups(nr, plain, rp, n_waves)]
        for fg in self._full_groups(nr, full, rf, n_waves, R):
            full_waves = self._kind_waves(2, fg, full, FULL_COST, nr, R)
            for pg, plain_waves in plains:
                waves = full_waves + plain_waves
                # the rest exchange the border rows, `border` jobs a side
                ex = min(n_waves - len(waves), max(1, 2 * border))
                if ex < 1 or border > tags or 2 * border > jobs * ex:
                    continue
                waves += [(EXCHANGE_COST, 0, 3, 0)] * ex
                waves += [(0.0, 0, 0, 0)] * (n_waves - len(waves))
                waves.sort(reverse=True)
                waves = waves[:4] + waves[4:][::-1]  # wave w runs on SIMD w % 4
                # waves w and w + 4 share a SIMD; a border that is late holds up
                # the neighbours too, so work beside an exchange wave counts more
                cost = max(a[0] * (EXCHANGE_SHARE if b[2] == 3 else 1.0) +
                           b[0] * (EXCHANGE_SHARE if a[2] == 3 else 1.0) for a, b in zip(waves[:4], waves[4:]))
                work = sum(w[0] for w in waves)
                key = (cost + STEP_COST + SHARE_COST * work, work)
                if best is None or key < best[0]:
                    best = (key, fg, pg, ex, [(k, t) for _, _, k, t in waves])
        self.ok = best is not None
        if self.ok:
            (self.cost, _), self.full_groups, self.plain_groups, self.exchange, self.waves = best

    @staticmethod
    def _counts(nr, cols, most, n_waves):
        """Numbers of row groups of at most ``most`` rows that differ in their
        size and fit the waves."""
        return sorted({-(-nr // k) for k in range(1, most + 1)} - {n for n in range(nr + 1) if n * cols > 64 * (n_waves - 1)})

    @classmethod
    def _full_groups(cls, nr, full, rf, n_waves, R):
        """Candidate splits: lists of row groups, each from a wave of its own."""
        if not full:
            return [[]]
        out = [[_border_first(_groups(nr, n))] for n in cls._counts(nr, full, rf, n_waves)]
        if R and nr > 2 * R:
            inner = nr - 2 * R
            for per in (1, 2):  # rows of a group at the border
                edge = [(r, min(per, R - r)) for r in range(0, R, per)]
                edge += [(nr - R + r, k) for r, k in edge]
                for n in cls._counts(inner, full, rf, n_waves):
                    out.append([edge, [(r + R, k) for r, k in _groups(inner, n)]])
        return out

    @classmethod
    def _plain_groups(cls, nr, plain, rp, n_waves):
        if not plain:
            return [[]]
        return [[_border_first(_groups(nr, n))] for n in cls._counts(nr, plain, rp, n_waves)]

    @staticmethod
    def _kind_waves(kind, parts, cols, unit, nr, R):
        """(work, rows that wait for a border, kind, first thread) of the waves
        that hold ``parts``, each part from a wave of its own."""
        out, t0 = [], 0
        for groups in parts:
            n = len(groups) * cols
            for w in range(-(-n // 64)):
                mine = groups[w * 64 // cols:(min(n, w * 64 + 64) - 1) // cols + 1]
                late = max(sum(x < R or x + R >= nr for x in range(r, r + k)) for r, k in mine)
                out.append((max(k for _, k in mine) * unit, late, kind, t0))
                t0 += 64
        return out


def _border_first(groups):
    """The first and the last group, then the others."""
    return groups[:1] + groups[:0:-1][:1] + groups[1:-1] if len(groups) > 2 else groups


def _copy_bytes(nr, nzc, full, hc, R, n_fcells):
    return (((nr + 2 * R) * (nzc + hc) + hc) * 16, (nr + 2 * R) * full * 16, (nr * (full + 2 * hc) + hc) * 16,
            n_fcells * 16)


def lds_copies(strips, hc, R, n_fcells):
    """Bytes of one copy of u, Phix, Phiz and the source cells of strips (an
    array of their numbers, or one strip's)."""
    return _copy_bytes(strips.T[2], strips.T[21], strips.T[4] + strips.T[5], hc, R, n_fcells)


def lds_offsets(copies, nr, itemsize):
    """Where Phix, Phiz, the source cells, the x profiles and the flags begin:
    u comes first, two copies each of all but the profiles."""
    return np.cumsum([2 * c for c in copies] + [-(-nr * 2 * itemsize // 16) * 16], axis=0)


def _split(total, rows, R):
    """(strips, rows, strips of one row more) of equal strips of at most
    ``rows`` rows, each at least R."""
    n = max(1, min(-(-total // rows), total // R if total >= R else 1))
    return (n,) + divmod(total, n)


class _Kept(object):
    """At most ``most`` values by key, the one used longest ago dropped first;
    several threads may ask at once (a value may then be made twice)."""

    def __init__(self, most):
        self.most = most
        self._lock = threading.Lock()
        self._kept = collections.OrderedDict()

    def get(self, key, make):
        with self._lock:
            if key in self._kept:
                self._kept.move_to_end(key)
                return self._kept[key]
        value = make()
        with self._lock:
            value = self._kept.setdefault(key, value)
            self._kept.move_to_end(key)
            while len(self._kept) > self.most:
                self._kept.popitem(last=False)
        return value

    def clear(self):
        with self._lock:
            self._kept.clear()

    def __len__(self):
        return len(self._kept)


_LAYOUTS = _Kept(4096)


class ShotStrips(object):
    """The ways to cut one shot into strips of at most ``most`` rows: its
    column split and, for a bound on the cost of a step, the strips (x0, rows,
    x type)."""

    def __init__(self, shape, pml, R, itemsize, limits, n_fcells_row, most):
        (xl, xr), (zl, zr) = pml
        self.nx, self.nz = shape
        self.most = most
        self.R, self.itemsize, self.limits = R, itemsize, limits
        self.V = 16 // itemsize
        self.hc = -(-R // self.V)
        self.nzc, self.zfl, self.zfr = z_columns(self.nz, zl, zr, R, self.V)
        left, right = max(xl, 1) + R, max(xr, 1) + R
        self.n_fcells_row = n_fcells_row
        if self.zfl == self.nzc or self.nx - left - right < max(R, 1):
            # all cells full anyway, or no room between the x sides
            self.segments = [(0, self.nx, True)]
        else:
            self.segments = [(0, left, True), (left, self.nx - left - right, False), (self.nx - right, right, True)]
        self._costs, self._ok, self._splits = {}, {}, {}

    def fits(self, nr, xtype):
        full = self.nzc if xtype else self.zfl + self.zfr
        copies = _copy_bytes(nr, self.nzc, full, self.hc, self.R, self.n_fcells_row * nr)
        return 2 * sum(copies) + -(-nr * 2 * self.itemsize // 16) * 16 + 32 <= LDS_BYTES

    def layout(self, nr, xtype, alone=False):
        full = self.nzc if xtype else self.zfl + self.zfr
        # jobs of a border: u over all cells and Phix over the full ones, 64
        # columns each
        border = -(-self.nzc // 64) - (-full // 64)
        key = (nr, self.nzc - full, full, self.limits, border, self.R, alone)
        return _LAYOUTS.get(key, lambda: Layout(*key))

    def costs(self, xtype):
        """(rows, cost) of the strips that fit a workgroup, by rows."""
        if xtype not in self._costs:
            out = []
            for nr in range(self.R, min(self.nx, self.most) + 1):
                if not self.fits(nr, xtype):
                    break
                lay = self.layout(nr, xtype)
                if lay.ok:
                    out.append((nr, lay.cost))
            self._costs[xtype] = out
        return self._costs[xtype]

    def split(self, bound, rows_z=None):
        """Strips that cost at most ``bound`` a step, or None: the fewest, but
        those away from the x PML of about ``rows_z`` rows if that is given;
        per segment (x0, x type, strips, rows, strips of one row more)."""
        if (bound, rows_z) not in self._splits:
            self._splits[bound, rows_z] = self._split(bound, rows_z)
        return self._splits[bound, rows_z]

    def _split(self, bound, rows_z):
        if self.fits(self.nx, True) and rows_z is None:
            lay = self.layout(self.nx, True, True)
            if lay.ok and lay.cost <= bound:
                return [(0, True, 1, self.nx, 0)]
        out = []
        for x0, total, xtype in self.segments:
            if (xtype, bound) not in self._ok:
                ok = [nr for nr, c in self.costs(xtype) if c <= bound]
                self._ok[xtype, bound] = ok[::-1], set(ok)
            order, ok = self._ok[xtype, bound]
            for rows in ([rows_z] if rows_z is not None and not xtype else order):
                n, nr, more = _split(total, rows, self.R)
                if nr in ok and (not more or nr + 1 in ok):
                    break
            else:
                return None
            out.append((x0, xtype, n, nr, more))
        return out

    def count(self, bound, rows_z=None):
        """The number of strips of ``split``, or None."""
        got = self.split(bound, rows_z)
        return None if got is None else sum(s[2] for s in got)

    def cut(self, bound, rows_z=None):
        """``split`` strip by strip, (x0, rows, x type), or None."""
        got = self.split(bound, rows_z)
        if got is None:
            return None
        out = []
        for x0, xtype, n, nr, more in got:
            for i in range(n):
                out.append((x0, nr + (i < more), xtype))
                x0 += out[-1][1]
        return out

    def bounds(self):
        """The costs a strip of this shot can have."""
        out = {c for _, _, xtype in self.segments for _, c in self.costs(xtype)}
        if self.fits(self.nx, True) and self.layout(self.nx, True, True).ok:
            out.add(self.layout(self.nx, True, True).cost)
        return out


def plan_groups(shots, cus):
    """The cost of a step and the consecutive shots that run together with
    their strips, a list of (shots, strip lists); None if a shot does not fit.  Of the ways to spread the
    shots evenly over the fewest groups, or one or two more, the one whose
    groups' steps cost least together; strips cost alike within a group."""
    bounds = sorted(set().union(*[s.bounds() for s in set(shots)]))
    if not bounds:
        return None

    def fill(group):
        """(bound, rows away from the x PML): the least bound whose strips fit
        the compute units and, where units are left, the lowest strips beside
        it.  Few may be as low as R rows; many exchange so many rows that those
        of less than 2 R, where every row waits for both borders, are slower
        (FP32, 1 shot: 1041 x 341 nodes of order 8, 6.6 us a step with 178
        strips and 6.0 with 123; 186 x 113 of order 8, 4.9 with 24 and 6.0 with
        19; 360 x 332 of order 4, 4.4 with 180 and 5.3 with 83)."""
        def count(*bound):
            c = [shots[i].count(*bound) for i in group]
            return cus + 1 if None in c else sum(c)
        lo, hi = 0, len(bounds) - 1
        if count(bounds[hi]) > cus:
            return None
        while lo < hi:
            mid = (lo + hi) // 2
            if count(bounds[mid]) <= cus:
                hi = mid
            else:
                lo = mid + 1
        n, R = count(bounds[lo]), max(shots[i].R for i in group)
        for first, most in ((R, min(3 * cus // 4, 2 * cus // R)), (2 * R, cus)):
            for rows in range(first, 4 * R):
                if n < count(bounds[lo], rows) <= most:
                    return bounds[lo], rows
        return (bounds[lo],)

    weight = [s.count(bounds[-1]) for s in shots]
    if any(f is None or f > cus for f in weight):
        return None
    total = sum(weight)
    best = None
    first = max(1, -(-total // cus))
    for n in range(first, len(shots) + 1):
        groups, load = [[] for _ in range(n)], 0
        for i, t in enumerate(weight):
            groups[min(n - 1, int((load + t / 2) * n / total))].append(i)
            load += t
        groups = [g for g in groups if g]
        got = [fill(g) for g in groups]
        if all(b is not None for b in got) and (best is None or sum(b[0] for b in got) < best[0]):
            best = (sum(b[0] for b in got), [(g, [shots[i].cut(*b) for i in g]) for g, b in zip(groups, got)])
        if best is not None and n >= first + 2:
            break
    return best


def thread_items(lay, xtype, nzc, zfl, zfr, R, limits):
    """(threads, 4) item table of a workgroup, and the owner of every cell:
    thread and march step, (rows, columns).  A lane left over in a wave repeats
    the cells of another thread, which its item names."""
    rp, rf, threads = limits[:3]
    items = np.zeros((threads, 4), dtype=np.int32)
    owner = np.full((lay.nr, nzc, 2), -1, dtype=np.int32)
    alias = np.arange(threads)
    full_cols = np.arange(nzc) if xtype else np.concatenate([np.arange(zfl), np.arange(nzc - zfr, nzc)])
    plain_cols = np.setdiff1d(np.arange(nzc), full_cols)
    for kind, cols, parts, RM in ((2, full_cols, lay.full_groups, rf), (1, plain_cols, lay.plain_groups, rp)):
        # thread t of the kind: its wave by the wave's first thread
        wave_of = {t0 // 64: w for w, (k, t0) in enumerate(lay.waves) if k == kind}
        t0 = 0
        for groups in parts:
            row0, size = (np.array(v) for v in zip(*groups))
            n = len(groups) * cols.size
            t = np.arange(-(-n // 64) * 64)
            live = t < n
            g = np.where(live, t // cols.size, len(groups) - 1)
            col, cnt, r0 = cols[t % cols.size], size[g], row0[g]
            # the group at the top marches towards it, unless it holds every row
            rev = (r0 == 0) & (cnt < lay.nr) & (cnt > 1)
            top, bot = r0 < R, r0 + cnt - 1 + R >= lay.nr
            # the border a march starts at is needed at once, the other at its end
            wait = np.where(top, np.where(rev, END_TOP, BEGIN_TOP), 0) | np.where(bot, np.where(rev, BEGIN_BOT, END_BOT), 0)
            flags = np.where(rev, REV, 0) | np.where(live, wait, 0) | KIND * kind
            rbase = np.where(rev, r0 + RM - 1, r0 - (RM - cnt))
            own = np.where(live, ((1 << RM) - 1) & ~((1 << (RM - cnt)) - 1), 0)
            first = (RM - cnt).reshape(-1, 64).min(axis=1).repeat(64)
            late = RM - cnt > first
            tids = np.array([wave_of[t0 // 64 + i] for i in t // 64]) * 64 + t % 64
            items[tids] = np.stack([rbase, flags, own | (first << 16) | (late.astype(np.int64) << 24), col], axis=1)
            for j in range(RM):
                m = ((own >> j) & 1) == 1
                row = rbase[m] + j * np.where(rev[m], -1, 1)
                owner[row, col[m], 0] = tids[m]
                owner[row, col[m], 1] = j
            alias[tids] = owner[r0, col, 0]
            t0 += t.size
    # the exchange waves know their number, the idle ones follow them
    for i, w in enumerate(sorted((w for w, (k, _) in enumerate(lay.waves) if k in (0, 3)),
                                 key=lambda w: -lay.waves[w][0])):
        items[64 * w:64 * w + 64, 0] = i
        items[64 * w:64 * w + 64, 1] = 3 * KIND
    items[:, 3] |= alias << 16
    return items, owner


# a plan holds 0.1 to 0.6 MB; a survey of shots of uneven aperture,
# modeled shot by shot, comes back to each of its plans (4 ms to make, 9 to 14
# those of 16 to 32 shots)
_PLANS = _Kept(256)


class Plan(object):
    """What the sizes of a batch's shots (``keys``: shape, PML widths and most
    source cells of a row) decide: the groups, the strips without their
    sources and receivers, and the thread tables of the kinds of strips.
    ``ok`` is False where a shot does not suit the loop."""

    @classmethod
    def of(cls, keys, R, itemsize, limits, cus):
        key = (keys, R, itemsize, limits, cus)
        # with the rule that groups the shots: a plan is kept for it alone
        return _PLANS.get((plan_groups,) + key, lambda: cls(*key))

    def __init__(self, keys, R, itemsize, limits, cus):
        groups = None
        # strips much higher than the compute units ask for are not looked at
        # unless the others do not do
        rows = max(16, 4 * -(-sum(k[0][0] for k in keys) // cus))
        for most in (rows, max(k[0][0] for k in keys)):
            memo = {k: ShotStrips(k[0], k[1], R, itemsize, limits, k[2], most) for k in set(keys)}
            groups = plan_groups([memo[k] for k in keys], cus)
            if groups is not None:
                break
        self.ok = groups is not None
        if not self.ok:
            return
        self.cost, groups = groups
        cuts = [memo[k] for k in keys]
        self.nzc = np.array([c.nzc for c in cuts])
        strips, templates = [], {}
        self.group_begin, self.first_strip = [0], []
        # per shot, which of the distinct cuts it has, and of these the strip of
        # every row: shots of one cut have the same strips
        self.cut_of, self.row_strip, known = [], [], {}
        for shots, cut in groups:
            for si, parts in zip(shots, cut):
                c = cuts[si]
                self.first_strip.append(len(strips))
                if (c, tuple(parts)) not in known:
                    known[c, tuple(parts)] = len(known)
                    self.row_strip.append(np.repeat(np.arange(len(parts)), [nr for _, nr, _ in parts]))
                self.cut_of.append(known[c, tuple(parts)])
                for i, (x0, nr, xtype) in enumerate(parts):
                    lay = c.layout(nr, xtype, len(parts) == 1)
                    key = (lay, xtype, c.nzc, c.zfl, c.zfr)
                    if key not in templates:
                        templates[key] = (len(templates), thread_items(lay, xtype, c.nzc, c.zfl, c.zfr, R, limits))
                    me = len(strips)
                    up, down = i > 0, i + 1 < len(parts)
                    d = [0] * STRIP_INTS
                    d[0:4] = si, x0, nr, XTYPE if xtype else 0
                    if up and xtype and parts[i - 1][2]:
                        d[3] |= PXTOP
                    if down and xtype and parts[i + 1][2]:
                        d[3] |= PXBOT
                    d[4:6] = (c.nzc, 0) if xtype else (c.zfl, c.zfr)
                    d[6:8] = c.zfl, c.zfr
                    d[19:24] = me - 1 if up else -1, me + 1 if down else -1, c.nzc, me, lay.exchange
                    d[28] = templates[key][0]
                    strips.append(d)
            self.group_begin.append(len(strips))
        self.strips = np.array(strips, dtype=np.int64)
        self.first_strip.append(len(strips))
        tables = [t for _, t in templates.values()]
        self.items = np.stack([t[0] for t in tables])
        # owners of the cells of all templates, (thread, step) a cell
        self.owner = np.concatenate([t[1].reshape(-1, 2) for t in tables])
        self.owner_base = np.cumsum([0] + [t[1].shape[0] * t[1].shape[1] for t in tables])


class ResidentTables(object):
    """Device tables of one batch for the resident loop (``build`` returns
    None where the batch does not suit it)."""

    @classmethod
    def plan(cls, shots, R, item, dev, always=False, nodes=None):
        """The plan of a batch of ``shots`` in its own order (``by_length``),
        or None where the step kernels take it: known before any table or
        state of the batch is made."""
        import torch
        most = cls._source_cells_per_row(shots, 16 // item, nodes)
        if not most or R not in (1, 2, 3, 4):
            return None
        limits = N.resident_limits()
        keys = tuple((tuple(int(n) for n in s.shape), tuple((l.size, r.size) for l, r in s.kpml), m)
                     for s, m in zip(shots, most))
        cus = torch.cuda.get_device_properties(dev).multi_processor_count
        plan = Plan.of(keys, R, item, limits, cus)
        if not plan.ok:
            return None
        # few nodes in costly strips (thick PML, FP64 of order 8) step faster
        # through the caches: 116 x 288 nodes in FP64 at cost 113 takes 11.1 us
        # here and 8.6 there, 104 x 104 (4 shots, cost 53) 10.9 and 9.2; at
        # cost 53, 448 x 175 in FP64 takes 11.8 and 12.0
        size = sum(k[0][0] * k[0][1] for k in keys)
        if not always and plan.cost > STEP_KERNEL_COST + size * item / STEP_KERNEL_BYTES:
            return None
        return plan

    @classmethod
    def build(cls, batch, always=False):
        """The tables of ``batch``, from its plan if the batch was made with
        one."""
        plan = batch._resident_plan
        if plan is None:
            plan = cls.plan(batch.shots, batch.R, batch.dtype.itemsize, batch.dev, always,
                            (batch.src_nodes, batch.adj_nodes))
        return None if plan is None else cls(batch, plan, N.resident_limits())

    @staticmethod
    def _source_cells_per_row(shots, V, nodes=None):
        """Per shot, the most source cells in any of its rows, forward or
        adjoint; None if one is not 2D, has no adjoint entries or has an entry
        off its grid (which a batch refuses).  ``nodes``: per way and shot the
        entries' flat nodes, where a batch has gathered them."""
        known, most = {}, []
        for si, s in enumerate(shots):
            if len(s.shape) != 2 or s.adj is None:
                return None
            nx, nz = s.shape
            cells = -(-nz // V)
            n = 0
            for way, (pos, _, _) in enumerate((s.src, s.adj)):
                key = (pos.__array_interface__["data"][0], pos.shape, pos.strides, nx, nz)
                if key not in known:
                    known[key] = 0
                    if pos.shape[0]:
                        x, z = np.divmod(nodes[way][si].node, nz) if nodes else (pos[:, 0], pos[:, 1])
                        x0, x1 = int(x.min()), int(x.max())
                        if x0 < 0 or x1 >= nx or z.min() < 0 or z.max() >= nz:
                            return None
                        some = np.zeros((x1 - x0 + 1, cells), dtype=bool)
                        some.reshape(-1)[(x - x0) * cells + z // V] = True
                        known[key] = int(np.count_nonzero(some, axis=1).max())
                n = max(n, known[key])
            most.append(n)
        return most

    def __init__(self, batch, plan, limits):
        import torch
        dev, R, item = batch.dev, batch.R, batch.dtype.itemsize
        V = 16 // item
        hc = -(-R // V)
        strips = plan.strips.copy()
        n = len(strips)
        # tables of the shots, made once for those that have the same entries
        # and the same cut
        known, ways, recs = {}, ([], []), []

        def once(make, of, si, *more):
            key = id(of), plan.cut_of[si], batch.shots[si].shape
            if key not in known:
                cut = plan.strips[plan.first_strip[si]:plan.first_strip[si + 1]]
                known[key] = make(plan, cut, plan.row_strip[plan.cut_of[si]], batch.shots[si].shape[1], of, *more)
            return known[key]

        for si in range(batch.n_shots):
            for way, nodes in enumerate((batch.src_nodes, batch.adj_nodes)):
                ways[way].append(once(self._sources, nodes[si], si, V))
            recs.append(once(self._receivers, batch.rec_nodes[si], si, batch.adj_nodes[si], R, hc, item))
        inj, fcells = [], np.zeros(n, dtype=np.int64)
        for way, nodes in enumerate((batch.src_nodes, batch.adj_nodes)):
            t = ways[way]
            base = np.cumsum([0] + [ne.node.size for ne in nodes])
            strips[:, 10 + 2 * way] = np.concatenate([b + x["first"][:-1] for b, x in zip(base, t)])
            strips[:, 11 + 2 * way] = np.concatenate([b + x["first"][1:] for b, x in zip(base, t)])
            fcells = np.maximum(fcells, np.concatenate([x["cells"] for x in t]))
            # blocks of thread tables, one copy for alike shots
            blocks, at, size = [], {}, 0
            for x in t:
                if id(x) not in at:
                    at[id(x)] = size
                    blocks.append(x["finfo"])
                    size += len(x["finfo"])
            strips[:, 29 + way] = np.concatenate([np.where(x["block"] < 0, -1, x["block"] + at[id(x)]) for x in t])
            finfo = np.concatenate(blocks) if size else np.zeros((1, limits[2], 2), dtype=np.int32)
            inj.append({"finfo": finfo, "lds": np.concatenate([x["lds"] for x in t])})
        strips[:, 24:28] = np.stack(lds_copies(strips, hc, R, fcells), axis=1)
        strips[:, 14:19] = lds_offsets(strips[:, 24:28].T, strips[:, 2], item).T
        # receiver nodes, in strip order
        base = np.cumsum([0] + [t["lds"].size for t in recs])
        strips[:, 8] = np.concatenate([b + t["first"][:-1] for b, t in zip(base, recs)])
        strips[:, 9] = np.concatenate([b + t["first"][1:] for b, t in zip(base, recs)])
        rec_lds = np.concatenate([t["lds"] for t in recs])
        rec_node = np.concatenate([t["node"] + np.int32(b) for b, t in zip(base, recs)])
        self.n_rec_nodes = int(base[-1])

        # one upload, every table from a multiple of 16 bytes on
        tables = [strips, plan.items, rec_lds, rec_node]
        for t in inj:
            tables += [t["finfo"], t["lds"]]
        at, size = [], 0
        for t in tables:
            at.append(size)
            size += -(-t.size // 4) * 4
        # (numpy: a tensor's fill wakes torch's threads, which then compete
        # with numpy's for milliseconds)
        flat = np.zeros(size + 4, dtype=np.int32)
        for a, t in zip(at, tables):
            flat[a:a + t.size] = t.reshape(-1)
        self._tables = torch.from_numpy(flat).to(dev)
        ptr = self._tables.data_ptr()
        # the nodes' entries {nptr, chan, w, shot}: the step kernels' tables
        # where these have every shot's nodes in ascending order
        self._entries = [inj[2:6] if by_node else self._node_entries(batch, nodes)
                         for inj, by_node, nodes in ((batch.fwd_inj, batch.src_by_node, batch.src_nodes),
                                                     (batch.adj_inj, batch.adj_by_node, batch.adj_nodes))]
        self.n_inj = [int(t["lds"].size) for t in inj]
        self.n_strips, self.cost = n, plan.cost
        self.group_begin = np.asarray(plan.group_begin, dtype=np.int32)
        self.group_lds = np.array([strips[a:b, 18].max() + 32 for a, b in zip(plan.group_begin[:-1], plan.group_begin[1:])],
                                  dtype=np.int32)
        cells = 2 * -(-int(strips[:, 21].max()) // 64) * 64 * R
        stride = 2 * limits[4] * 4 + 4 * cells * 16
        self.xchg = torch.zeros(n * stride // 4, dtype=torch.int32, device=dev)
        own = [t for way, by_node in zip(self._entries, (batch.src_by_node, batch.adj_by_node)) if not by_node for t in way]
        self._fixed = sum(t.numel() * t.element_size() for t in [self._tables, self.xchg] + own)
        self.epoch = ctypes.c_uint(0)
        self._work, self._item = None, item
        self.slot_bytes = max(1, self.n_inj[0] + self.n_rec_nodes, self.n_inj[1]) * item
        # bytes of working space under a memory budget (DeviceBatch.plan_segments)
        self.room = 0
        q = self.struct = N.Resident()
        q.n_strips, q.n_groups = n, len(self.group_lds)
        q.group_begin = self.group_begin.ctypes.data
        q.group_lds = self.group_lds.ctypes.data
        q.strips, q.items, q.rec_lds, q.rec_node = (ptr + 4 * a for a in at[:4])
        for way in range(2):
            q.finfo[way], q.inj_lds[way] = (ptr + 4 * a for a in at[4 + 2 * way:6 + 2 * way])
            q.inj_nptr[way], q.inj_chan[way], q.inj_w[way], q.inj_shot[way] = (t.data_ptr() for t in self._entries[way])
            q.n_inj[way] = self.n_inj[way]
        q.n_rec_nodes = self.n_rec_nodes
        q.xchg, q.xchg_stride, q.xchg_cells = self.xchg.data_ptr(), stride, cells
        q.spin = SPIN
        self.err = _WORDS.take(self)
        q.err = self.err.data_ptr()
        self._stop = torch.zeros(1, dtype=torch.int32, device=dev)
        q.stop = self._stop.data_ptr()
        q.epoch = ctypes.addressof(self.epoch)

    @staticmethod
    def _node_entries(batch, nodes):
        """Device arrays {nptr, chan, w, shot} of the nodes' entries."""
        base = np.cumsum([0] + [ne.chan.size for ne in nodes])
        nptr = np.concatenate([b + ne.nptr[:-1] for b, ne in zip(base, nodes)] + [base[-1:]])
        shot = np.repeat(np.arange(len(nodes)), [ne.node.size for ne in nodes])
        return batch._send([(np.int32, [nptr]), (np.int32, [ne.chan for ne in nodes]),
                            (np.float64, [ne.w for ne in nodes]), (np.int32, [shot])])

    @staticmethod
    def _sources(plan, strips, row_strip, nz, nodes, V):
        """Source tables of one shot with these ``strips``: where a node's
        value lies among its strip's source cells (``lds``); per strip the
        first of its nodes and its source cells; for the strips with sources
        (``block``: their number, or -1), per thread the first source cell and
        the march steps that have one (``finfo``)."""
        n, threads = len(strips), plan.items.shape[1]
        x, z = np.divmod(nodes.node, nz)
        st = row_strip[x]
        row = x - strips[st, 1]
        own = plan.owner[plan.owner_base[strips[st, 28]] + row * strips[st, 21] + z // V]
        # a strip's cells in the order its threads march over them
        key = (st * threads + own[:, 0]) * 64 + own[:, 1]
        cells, inv = np.unique(key, return_inverse=True)
        owner, step = cells // 64, cells % 64
        begin = np.searchsorted(owner // threads, np.arange(n + 1))
        some = np.nonzero(begin[1:] > begin[:-1])[0]
        block = np.full(n, -1)
        block[some] = np.arange(some.size)
        finfo = np.zeros((some.size, threads, 2), dtype=np.int32)
        if some.size:
            heads = np.nonzero(np.concatenate([[True], owner[1:] != owner[:-1]]))[0]
            k, t = np.divmod(owner[heads], threads)
            finfo[block[k], t, 0] = heads - begin[k]
            finfo[block[k], t, 1] = np.bitwise_or.reduceat(1 << step, heads)
        return {"lds": (inv.reshape(-1) - begin[st]) * V + z % V, "first": np.searchsorted(st, np.arange(n + 1)),
                "finfo": finfo, "block": block, "cells": np.diff(begin)}

    @staticmethod
    def _receivers(plan, strips, row_strip, nz, rec, adj, R, hc, item):
        """Receiver tables of one shot with these ``strips``: where a node
        lies in LDS, the first node of every strip, and the node of every
        entry (flat nodes ``rec``, in most batches those of the adjoint
        entries ``adj``)."""
        if np.array_equal(rec, adj.given):
            node, of = adj.node, adj.rank()
        else:
            node, of = np.unique(rec, return_inverse=True)
            of = of.reshape(-1).astype(np.int32)
        x, z = np.divmod(node, nz)
        st = row_strip[x]
        lds = (R + x - strips[st, 1]) * (strips[st, 21] + hc) * 16 + hc * 16 + z * item
        return {"lds": lds, "first": np.searchsorted(st, np.arange(len(strips) + 1)), "node": of}

    def chunk_slots(self, max_nt, room):
        """Slots of a run of ``max_nt`` that are worked on at a time: what
        ``room`` bytes hold of source values and receiver nodes, or
        CHUNK_LEAST."""
        return min(max_nt, max(CHUNK_LEAST, min(CHUNK_SLOTS, room // self.slot_bytes)))

    def reserve(self, max_nt, room):
        """Bytes that the loop takes beside the batch's state and stores in
        runs of up to ``max_nt`` slots: tables, border rows, working space in
        ``room`` bytes, and the sources of a run too short for the loop."""
        short = self.n_inj[1] * min(max_nt, RESIDENT_MIN_SLOTS - 1) * self._item
        return self._fixed + self.slot_bytes * self.chunk_slots(max_nt, room) + short

    def held(self):
        """Bytes of what ``reserve`` counts that are allocated."""
        return self._fixed + (self._work[0] * self.slot_bytes if self._work else 0)

    def release(self):
        """Give the working space back once the current stream is done with
        it (its own stream may be another); the next run takes it again."""
        import torch
        if self._work is not None:
            self._work[1].record_stream(torch.cuda.current_stream())
        self._work = None

    def _workspace(self, batch):
        """Source values and receiver nodes of a chunk of slots, one behind
        the other: a forward run has few sources, an adjoint no receivers."""
        import torch
        slots = self.chunk_slots(batch.max_nt, CHUNK_BYTES if batch.memory_budget is None else min(CHUNK_BYTES, self.room))
        have = self._work[0] if self._work else 0
        # a larger one stays where nothing bounds it (the time axis may change again)
        if have < slots or (have > slots and batch.memory_budget is not None):
            # first: both together may not fit, nor this and a long run's sources for the step kernels
            self.release()
            if batch.memory_budget is not None:
                batch.release_sources()
            self._work = slots, torch.empty(slots * self.slot_bytes // self._item, dtype=batch.tdtype, device=batch.dev)
        slots, work = self._work
        q = self.struct
        q.pre_slots = q.rec_slots = slots
        q.pre = work.data_ptr()
        q.recbuf = work.data_ptr() + slots * self.n_inj[0] * self._item

    def expired(self):
        """Whether a wait for a neighbour ran into its bound in a run that the
        host knows of: all those before the last time it waited for them."""
        return int(self.err[0]) != 0

    def seal(self, b, stream):
        """Behind the runs of a forward or an adjoint: NaN into the batch
        descriptor's traces and image if a wait expired in any of them."""
        N.call("pysit_amd_resident_seal", ctypes.byref(b), ctypes.byref(self.struct), stream)

    def run(self, batch, b, mode, j0, j1, direction, seg_base, record, stream):
        self._workspace(batch)
        if self.epoch.value > 0xF0000000:
            # the step tags wrap: start again from a cleared buffer
            self.xchg.zero_()
            self.epoch.value = 0
        N.call("pysit_amd_resident_run", ctypes.byref(b), ctypes.byref(self.struct), mode, j0, j1, direction,
               seg_base, 1 if record else 0, stream)
