"""The sub-tile MIC(0) sweeps' index arithmetic, restated on the CPU (no GPU):
the loader wave, the ring, the exchange planes and the PCG forms' fifth wave of
k_sweep_sub (libwetcloth_amd/csrc/wc_sweep.hip).  The mail records and the store
wave are in test_sweep_mail_addresses.py.

k_sweep_sub runs each 8x8 quarter of a 16x16 tile of the skewed box layout as
one unit, on the tile's steps from 8 (sa + sb) on.  Checked over box shapes, both
passes and both value types:
  - every address the loader forms, over all batches it reads ahead, is in the
    box and 16-byte aligned, and its loads fill each ring place once with the
    slot that belongs there (also with the steps' clamp taken out: then
    addresses leave the box, so the check is sharp);
  - the ring place a compute lane reads at step w holds the slot of its pencil's
    cell of that step;
  - no batch of the ring is read before it is complete or overwritten while a wave
    may still read it, and the load counter's waits fit its 6 bits;
  - between two barriers no wave touches a cell of the exchange planes that
    another one writes, and the operands are the neighbours' and halo cells;
  - the fifth wave updates every slot of r that a unit's steps hold once, and
    writes the x-face columns where k_face_cols puts them;
  - a unit's upstream units hold earlier tickets.
"""
import itertools

import numpy as np
import pytest

KT = 16
THREADS = KT * KT
KS = 8
KNB = 4
KPLANES = 8
ROW = KT + 1  # exchange-plane row stride
PLANE = ROW * ROW
CELL = {8: 32, 4: 16}  # bytes of a factor record by the value's

SHAPES = [(1, 1, 1), (8, 9, 3), (17, 7, 2), (16, 41, 7), (32, 25, 9), (40, 31, 16), (24, 33, 33)]
both = pytest.mark.parametrize("bwd", [False, True])
words = pytest.mark.parametrize("word", [4, 8])


class Ring:
    def __init__(self, word, pcg_forward=False, bwd=False):
        cell, rhs, op = (KNB * 64 * b // 1024 for b in (CELL[word], word, 4))
        self.batches = 64 * 1024 // (KNB * 64 * CELL[word])
        a = self.batches - 1
        while (a - 1) * (cell + 2 * rhs + op) > 63:
            a -= 1
        self.ahead = a
        self.loads = cell + rhs + op + (rhs if bwd or pcg_forward else 0)
        self.early = 1 if pcg_forward else 0


class Box:
    """An ex x ey x Bz box of DOFs in whole tiles, and its units."""

    def __init__(self, ex, ey, Bz):
        self.nua, self.nub = -(-ex // KS), -(-ey // KS)
        self.nta, self.ntb = -(-ex // KT), -(-ey // KT)
        self.Bz, self.nsteps = Bz, Bz + 2 * (KT - 1)
        self.ncell = self.nta * self.ntb * self.nsteps * THREADS
        self.nb = (Bz + 2 * (KS - 1) + KNB - 1) // KNB

    def units(self, bwd):
        for ub, ua in itertools.product(range(self.nub), range(self.nua)):
            yield Unit(self, ua, ub, bwd)


class Unit:
    def __init__(self, P, ua, ub, bwd):
        self.P, self.bwd, self.ua, self.ub = P, bwd, ua, ub
        A = ua + (2 * P.nta - P.nua if bwd else 0)
        B = ub + (2 * P.ntb - P.nub if bwd else 0)
        self.sa, self.sb = A & 1, B & 1
        self.a = P.nta - 1 - (A >> 1) if bwd else A >> 1
        self.b = P.ntb - 1 - (B >> 1) if bwd else B >> 1
        self.psa, self.psb = (1 - self.sa, 1 - self.sb) if bwd else (self.sa, self.sb)
        self.w0 = KS * (self.sa + self.sb)
        self.wend = P.nsteps - self.w0
        self.tile0 = (self.b * P.nta + self.a) * P.nsteps * THREADS

    def slot(self, w, p, clamp=True):
        """Slot of physical position p at the unit's step w (arrays)."""
        P = self.P
        wc = np.where(w < self.wend, self.w0 + w, P.nsteps - 1) if clamp else self.w0 + w
        wp = P.nsteps - 1 - wc if self.bwd else wc
        return (self.tile0 + wp * THREADS + (KS * self.psb + (p >> 3)) * KT + KS * self.psa +
                (p & 7))

    def pencil(self, lane):
        """(li, lj) of compute lane in the sweep's frame."""
        return KS * self.sa + (lane & 7), KS * self.sb + (lane >> 3)

    def cell(self, lane):
        """Its cell in an exchange plane."""
        li, lj = self.pencil(lane)
        return (lj + 1) * ROW + li + 1


def stream(E):
    """One array's loads of a batch: (step, position, byte in the ring) per
    16-byte piece; E: element size."""
    per = 1024 // (64 * E)
    lanes = 64 // per
    j, lane = np.divmod(np.arange(KNB // per * 64), 64)
    return j * per + lane // lanes, lane % lanes * (16 // E), j * 1024 + lane * 16


def records(E):
    """The same for the factor records, which may span pieces."""
    pieces = E // 16
    st, h, lane = np.unravel_index(np.arange(KNB * pieces * 64), (KNB, pieces, 64))
    return st, h * (64 // pieces) + lane // pieces, st * 64 * E + h * 1024 + lane * 16


@both
@words
def test_loader(bwd, word):
    outside = 0
    for shape in SHAPES:
        P = Box(*shape)
        ahead = Ring(word).ahead
        for u in P.units(bwd):
            for E, (st, p, at) in ((word, stream(word)), (4, stream(4)),
                                   (CELL[word], records(CELL[word]))):
                # the pieces fill [step][position] of the ring once, in order
                assert sorted(at) == list(range(0, KNB * 64 * E, 16))
                assert np.array_equal(at // E, st * 64 + p)
                for n in range(P.nb + ahead):
                    s = u.slot(n * KNB + st, p)
                    byte = s * E + at % E
                    assert s.min() >= 0 and (byte + 16).max() <= P.ncell * E
                    assert (byte % 16 == 0).all()
                    # a piece of smaller elements holds the following slots
                    if E < 16:
                        for k in range(16 // E):
                            assert np.array_equal(u.slot(n * KNB + st, p + k), s + k)
                    s = u.slot(n * KNB + st, p, clamp=False)
                    outside += int(((s < 0) | (s >= P.ncell)).any())
    assert outside


@both
def test_ring_position_matches_compute_lane(bwd):
    """Position lane (forward) or 63 - lane (backward) of step w is the slot of
    the lane's pencil on that step, whose cell is w - ui - uj."""
    for shape in SHAPES:
        P = Box(*shape)
        w = np.arange(P.nb * KNB)
        for u in P.units(bwd):
            w_in = w[w < u.wend]
            assert len(w_in) >= P.Bz + 2 * (KS - 1)
            for lane in range(64):
                li, lj = u.pencil(lane)
                s = u.slot(w_in, 63 - lane if bwd else lane)
                lane_s, step = s % THREADS, s // THREADS % P.nsteps
                lip, ljp = (KT - 1 - li, KT - 1 - lj) if bwd else (li, lj)
                assert (lane_s == ljp * KT + lip).all()
                kk = step - lip - ljp  # the physical cell
                if bwd:
                    kk = P.Bz - 1 - kk
                assert np.array_equal(kk, w_in - (lane & 7) - (lane >> 3))


@words
@pytest.mark.parametrize("form", ["forward", "pcg forward", "backward"])
def test_ring_order(word, form):
    """Interval n is the time between the barriers that hand over batches n and
    n + 1 (-1 and, with r's update, -2 before the loop)."""
    R = Ring(word, form == "pcg forward", form == "backward")
    assert 2 <= R.ahead < R.batches and (R.ahead - 1) * R.loads <= 63
    for nb in (4, 5, 9, 40):
        # complete[m]: the first interval that may read batch m
        complete, wait = {}, [(-1 - R.early, R.ahead - 1 - R.early, R.ahead)]
        wait += [(n, R.ahead - 2 - R.early, R.ahead + n) for n in range(nb)]
        for interval, flying, issued in wait:
            assert 0 <= flying * R.loads <= 63
            for m in range(issued - flying):
                complete.setdefault(m, interval)
        overwritten = {n + R.ahead - R.batches: n for n in range(nb)}  # by issue(n + ahead)
        for m in range(nb):
            reads = [m - 1, m]  # the compute wave; the store wave (r of z . r)
            if R.early:
                reads.append(max(m - 2, -2))  # r's update, of batches 0 and 1 before the loop
                if m == 1:
                    reads.append(-2)
            assert min(reads) >= complete[m]
            assert max(reads) < overwritten.get(m, 10 ** 9)


def plane_accesses(u, n, planes):
    """Cells of the exchange planes that each wave reads and writes in interval n
    of an unending unit."""
    own = [u.cell(lane) for lane in range(64)]
    at = lambda w, c: w % planes * PLANE + c
    acc = {k: (set(), set()) for k in ("compute", "face", "store")}
    for st in range(KNB):
        w = n * KNB + st
        for c in own:  # operands: x, y, z neighbours or the +0 at [0][0]
            acc["compute"][0].update(at(w - 1, c - d) for d in (1, ROW, 0, c))
            acc["compute"][1].add(at(w, c))
        w += KNB  # the face wave publishes the next batch's halos
        for m in range(KS):
            li, lj = KS * u.sa, KS * u.sb
            acc["face"][1].add(at(w - 1, (lj + m + 1) * ROW + li))
            acc["face"][1].add(at(w - 1, lj * ROW + li + m + 1))
        w -= 2 * KNB  # the store (and the column) wave read the last batch
        acc["store"][0].update(at(w, c) for c in own)
    return acc


def conflicts(u, planes):
    bad = 0
    for n in range(8, 12):
        acc = plane_accesses(u, n, planes)
        for p, q in itertools.permutations(acc, 2):
            bad += len(acc[p][1] & (acc[q][0] | acc[q][1]))
        assert all(c % PLANE for _, w in acc.values() for c in w)  # [0][0] stays +0
    return bad


def test_planes_between_barriers():
    P = Box(32, 32, 8)
    units = [u for u in P.units(False) if u.a == 0 and u.b == 0]
    assert {(u.sa, u.sb) for u in units} == {(0, 0), (0, 1), (1, 0), (1, 1)}
    for u in units:
        assert conflicts(u, KPLANES) == 0
        assert conflicts(u, KNB) > 0  # one batch's planes would not do


def test_plane_halos_are_the_operands():
    for sa, sb in itertools.product((0, 1), (0, 1)):
        u = next(u for u in Box(32, 32, 1).units(False) if (u.sa, u.sb) == (sa, sb))
        halo_x = {(KS * sb + m + 1) * ROW + KS * sa for m in range(KS)}
        halo_y = {KS * sb * ROW + KS * sa + m + 1 for m in range(KS)}
        own = {u.cell(lane): lane for lane in range(64)}
        for c, lane in own.items():
            assert (c - 1 in halo_x) if lane & 7 == 0 else own[c - 1] == lane - 1
            assert (c - ROW in halo_y) if lane >> 3 == 0 else own[c - ROW] == lane - 8
        assert not set(own) & (halo_x | halo_y) and 0 not in halo_x | halo_y


def test_residual_update_covers_r_once():
    for shape in SHAPES:
        P = Box(*shape)
        count = np.zeros(P.ncell, dtype=int)
        for u in P.units(False):
            for n, st in itertools.product(range(P.nb), range(KNB)):
                w = n * KNB + st
                if w < u.wend:
                    np.add.at(count, u.slot(w, np.arange(64)), 1)
        assert count.max() == 1
        assert (count[cells(P)] == 1).all()


def cells(P):
    """Slots of the cells of the units' pencils."""
    s = np.arange(P.ncell)
    lane, step, tile = s % THREADS, s // THREADS % P.nsteps, s // THREADS // P.nsteps
    x, y = tile % P.nta * KT + lane % KT, tile // P.nta * KT + lane // KT
    kk = step - lane % KT - lane // KT
    return (x < P.nua * KS) & (y < P.nub * KS) & (kk >= 0) & (kk < P.Bz)


def test_face_columns():
    for shape in SHAPES:
        P = Box(*shape)
        col = {0: {}, 15: {}}  # column index -> (unit, step, plane cell)
        for u in P.units(True):
            base = (u.tile0 >> 4)
            for n, lane in itertools.product(range(P.nb), range(KNB * KS)):
                w, row = n * KNB + lane // KS, lane % KS
                if w >= u.wend:
                    continue
                i = base + KS * u.psb + row + (P.nsteps - 1 - u.w0 - w) * KT
                own = 63 - (row * KS + (KS - 1 if u.psa else 0))
                side = col[15 if u.psa else 0]
                assert 0 <= i < P.ncell // KT and i not in side
                side[i] = True
                # the slot of that column entry is the plane cell's pencil and step
                t = i * KT + (15 if u.psa else 0)
                assert t == u.slot(w, 63 - own)
                li, lj = u.pencil(own)
                assert (t % THREADS % KT, t % THREADS // KT) == (KT - 1 - li, KT - 1 - lj)
        s = np.flatnonzero(cells(P))
        for x in (0, 15):  # every cell on a tile's x faces is written
            assert {int(t) >> 4 for t in s[s % KT == x]} <= set(col[x])


@both
def test_tickets_respect_dependencies(bwd):
    for shape in SHAPES:
        P = Box(*shape)
        order = [(A, s - A) for s in range(P.nua + P.nub - 1) for A in range(P.nua)
                 if 0 <= s - A < P.nub]
        ticket = {u: t for t, u in enumerate(order)}
        assert sorted(order) == sorted((u.ua, u.ub) for u in P.units(bwd))
        for (A, B), t in ticket.items():
            assert A == 0 or ticket[(A - 1, B)] < t
            assert B == 0 or ticket[(A, B - 1)] < t
